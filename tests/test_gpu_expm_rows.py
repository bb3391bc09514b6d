"""exp(X) by the series over dense rows against the series over pair products ("product_dense" = 0): the same offsets,
number of terms and exponent, and the same values -- every element is the same sum, so without squarings the same
numbers -- at the edges of the row kernel's workgroups, with overshot batches, few iterations and values that are not
finite."""
import ctypes

import numpy as np
import pytest

import diaq_amd  # noqa: F401  (registers diaq_gpu)

pytestmark = pytest.mark.gpu


def matrix(n, offs, norm, precision, seed=0, nan=False):
    import diaq_gpu as d
    rng = np.random.default_rng(n + 31 * seed)
    vals = [rng.standard_normal(n - abs(o)) + 1j * rng.standard_normal(n - abs(o)) for o in offs]
    for k, v in enumerate(vals):  # zero parts and zero blocks
        if k % 3 == 1:
            v.real = 0
        if k % 4 == 2:
            v[len(v) // 3: 2 * len(v) // 3] = 0
    if nan:
        vals[0][len(vals[0]) // 2] = np.nan
    scale = norm / sum(np.max(np.abs(np.nan_to_num(v))) for v in vals)
    return d.to_device(d.diaQMatrix.from_diagonals([n, n], offs, [v * scale for v in vals]), precision)


def expm(A, dense, t, max_iterations=100, tolerance=1e-12, cutoff=1.0):
    """(offsets, values by offset), terms and exponent of exp(-iAt)."""
    from diaq_amd import capi
    L, terms, s, out = capi.lib(), ctypes.c_int(), ctypes.c_int(), ctypes.c_void_p()
    capi.check(L.dq_set_tuning(b"product_dense", dense))
    try:
        capi.check(L.dq_expm_negative_taylor_scaled(A.handle, t, max_iterations, cutoff, tolerance, ctypes.byref(out),
                                                    ctypes.byref(terms), ctypes.byref(s)))
    finally:
        capi.check(L.dq_set_tuning(b"product_dense", 1))
    rows, k = ctypes.c_uint32(), ctypes.c_int32()
    capi.check(L.dq_devmat_info(out, ctypes.byref(rows), None, ctypes.byref(k), None, None))
    offs = np.zeros(k.value, np.int32)
    capi.check(L.dq_devmat_offsets(out, offs.ctypes.data_as(ctypes.POINTER(ctypes.c_int32))))
    starts = np.concatenate([[0], np.cumsum(rows.value - np.abs(offs.astype(np.int64)))])
    v = np.zeros((2, starts[-1]))
    pd = ctypes.POINTER(ctypes.c_double)
    capi.check(L.dq_devmat_download(out, starts[:-1].copy().ctypes.data_as(ctypes.POINTER(ctypes.c_int64)),
                                    v[0].ctypes.data_as(pd), v[1].ctypes.data_as(pd)))
    L.dq_devmat_destroy(out)
    return (list(offs), v), terms.value, s.value


def offsets(n, k, seed):
    r = np.random.default_rng(seed)
    return sorted(int(o) for o in r.choice(np.arange(-n + 1, n), size=min(k, 2 * n - 1), replace=False))


CASES = [(2, 3), (5, 4), (64, 9), (255, 70), (256, 5), (257, 5), (512, 6), (513, 66), (1024, 7), (1025, 7), (2047, 40),
         (2049, 40), (4097, 60)]


@pytest.mark.parametrize("n,k", CASES)
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_series_without_squarings(n, k, precision):
    if n > 2048 and precision == "fp32":
        pytest.skip("the large sizes in one precision")
    A = matrix(n, offsets(n, k, n), 0.6, precision)
    (U, m, s), (V, mv, sv) = expm(A, 1, 0.9), expm(A, 0, 0.9)
    assert (m, s) == (mv, sv) and s == 0
    assert U[0] == V[0]
    np.testing.assert_array_equal(U[1], V[1])


@pytest.mark.parametrize("n,k,t", [(3, 3, 3.0), (33, 5, 5.0), (100, 30, 3.0), (511, 9, 3.0), (513, 6, 6.0),
                                   (1030, 12, 3.0), (2050, 70, 1.8)])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_squarings(n, k, t, precision):
    A = matrix(n, offsets(n, k, n), 1.0, precision)
    (U, m, s), (V, mv, sv) = expm(A, 1, t, cutoff=0.2), expm(A, 0, t, cutoff=0.2)
    assert (m, s) == (mv, sv) and s >= 1
    assert U[0] == V[0]
    # |U| <= e^t; the terms' own rounding (the same on both sides in FP32) plus that of s squarings of up to n products
    tol = np.exp(t) * 2.0 ** s * (1e-13 if precision == "fp64" else 4 * 2.0 ** -24)
    np.testing.assert_allclose(U[1], V[1], rtol=0, atol=tol)


@pytest.mark.parametrize("offs", [[20, 30], [-30, -20], [-1, 20], [1, 2]])
@pytest.mark.parametrize("tolerance", [1e-12, 1e-3, 0.5])
def test_stops_inside_a_batch(offs, tolerance):
    A = matrix(64, offs, 0.8, "fp64")
    (U, m, s), (V, mv, sv) = expm(A, 1, 1.0, 100, tolerance), expm(A, 0, 1.0, 100, tolerance)
    assert (m, s) == (mv, sv)
    assert U[0] == V[0]
    np.testing.assert_array_equal(U[1], V[1])


@pytest.mark.parametrize("iterations", [0, 1, 5, 6, 7, 9])
def test_iteration_limit(iterations, capfd):
    A = matrix(70, [-3, 0, 2], 0.45, "fp64")
    out = []
    for dense in (1, 0):
        U, m, _ = expm(A, dense, 1.0, iterations)
        ctypes.CDLL(None).fflush(None)
        out.append((m, U[0], U[1], capfd.readouterr().out))
    assert out[0][:2] == out[1][:2] and out[0][3] == out[1][3]
    np.testing.assert_array_equal(out[0][2], out[1][2])


@pytest.mark.parametrize("nan,norm", [(True, 0.5), (False, 1e200)])
def test_not_finite(nan, norm):
    """Terms that are not finite (or overflow, where a large cutoff leaves them unscaled) keep to the pair products."""
    A = matrix(40, [-2, 0, 5], norm, "fp64", nan=nan)
    (U, m, s), (V, mv, sv) = (expm(A, dense, 1.0, 20, cutoff=1e300) for dense in (1, 0))
    assert (m, s) == (mv, sv)
    assert U[0] == V[0]
    np.testing.assert_array_equal(U[1], V[1])


@pytest.mark.parametrize("n", [1, 31, 32, 33, 65, 129, 300])
def test_small_products(n):
    """Near-dense powers at the edges of the small product's tiles."""
    import diaq_gpu as d
    rng = np.random.default_rng(n)
    M = (rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n))) / n
    got = d.to_numpy(d.pow(d.from_numpy(M), 4))
    ref = np.linalg.matrix_power(M, 4)
    # three products of length n: n eps times the product of the absolute values
    bound = np.linalg.matrix_power(np.abs(M), 4)
    assert np.all(np.abs(got - ref) <= 16 * n * 2.0 ** -53 * bound + 1e-300)


@pytest.mark.parametrize("n,near,a,cutoff,batches", [(4100, (1, 7, 49, 343, 1201, 2401), 11.0, 15.0, 1),
                                                     (4096, (1, 7, 61, 500, 1777), 20.0, 30.0, 2)])
def test_squaring_by_more_terms_than_a_batch(n, near, a, cutoff, batches):
    """A large cutoff leaves exp(-iAt/2) more terms than a batch of 32 (one row to a workgroup) or two (two rows), and the
    squaring applies them all at once: U V against SciPy's action of the exponential on V."""
    import diaq_gpu as d
    import scipy.sparse as sp
    from scipy.sparse.linalg import expm_multiply
    offs = sorted({0, *near, *(-o for o in near)})
    vals = [np.full(n - abs(o), 1.0 / len(offs)) for o in offs]
    A = d.to_device(d.diaQMatrix.from_diagonals([n, n], offs, [v + 0j for v in vals]), "fp64")
    (uo, uv), m, s = expm(A, 1, 2 * a, tolerance=1e-10, cutoff=cutoff)
    assert s == 1 and m > 32 * batches and 5 * m * len(offs) < n  # by terms, past the batches
    V = np.random.default_rng(n).choice([-1.0, 1.0], size=(n, 4))
    got, at = np.zeros((n, 4), complex), 0
    for o in uo:
        k = n - abs(o)
        r, c = max(0, -o), max(0, o)
        got[r:r + k] += (uv[0][at:at + k] + 1j * uv[1][at:at + k])[:, None] * V[c:c + k]
        at += k
    ref = expm_multiply(sp.diags(vals, offs, format="csr") * (-2j * a), V)
    # term k of a row carries k (diagonals + 3) roundings of a^k / k!: a (diagonals + 3) e^a eps for the series, twice that
    # through the second application, and its own; the truncation is below the tolerance
    assert np.max(np.abs(got - ref)) < 3 * a * (len(offs) + 3) * np.exp(a) * 2.0 ** -53 + 1e-9
