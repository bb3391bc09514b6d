"""The pair product's zero blocks (64 rows, real and imaginary part apart) and the map that a large result keeps: the bits
of the forms that read every value, with odd rows, diagonals that end inside a block and offsets that are no multiple of
a block; a NaN or infinity of x meets the result's zeros as without a map; new values replace the map."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from oracle import oracle as O  # noqa: E402

ROWS = 130001


def matrix(real):
    """24 diagonals whose blocks are zero on runs of 64 to 4096 rows, in one part or both."""
    rng = np.random.default_rng(5)
    offs = sorted({0, 1, -1, 63, -64, 128, 200, -513, 1024, -2048, 4100, -8192, 16384, -16385, 32768, -40000, 50001, 60000,
                   -60001, 129990, -129999, 7, 3000, -12345})
    vals = []
    for k, o in enumerate(offs):
        n = O.diagonal_length(o, ROWS, ROWS)
        r = np.arange(n) + max(0, -o)
        v = rng.standard_normal(n) + (0j if real else 1j * rng.standard_normal(n))
        if k % 3:
            v = v * (r // (64 << (k % 7)) % 2)
        if k % 5 == 4 and not real:
            v = np.where(r // 128 % 2, v.real + 0j, 1j * v.imag)
        vals.append(v)
    return O.Dia(ROWS, ROWS, offs, vals)


def tuning(key, value):
    from diaq_amd import capi
    capi.check(capi.lib().dq_set_tuning(key, value))


def spmv(C, x):
    import diaq_gpu as d
    import torch
    xr, xi = (torch.as_tensor(p, device="cuda").contiguous() for p in (x.real, x.imag))
    yr, yi = torch.empty_like(xr), torch.empty_like(xi)
    d.spmv_device(C, xr.data_ptr(), xi.data_ptr(), yr.data_ptr(), yi.data_ptr(), 0)
    torch.cuda.synchronize()
    return yr.cpu().numpy(), yi.cpu().numpy()


@pytest.mark.parametrize("real", [True, False])
def test_product_of_zero_blocks(real):
    import diaq_amd  # noqa: F401
    import diaq_gpu as d
    import torch
    from diaq_amd import capi
    M = matrix(real)
    D = d.to_device(d.diaQMatrix.from_diagonals([ROWS, ROWS], M.offsets, M.vals))
    got = {}
    try:
        for rpt in (0, 4, 16):
            tuning(b"product_rows_per_lane", rpt)
            got[rpt] = d.product(D, D)
        tuning(b"product_rows_per_lane", 0)
        tuning(b"product_skip_zero_blocks", 0)
        plain = d.product(D, D)
    finally:
        tuning(b"product_rows_per_lane", 0)
        tuning(b"product_skip_zero_blocks", 1)
    assert 16 * plain.stored > 1 << 28  # large enough to keep a map
    rng = np.random.default_rng(6)
    x = rng.standard_normal(ROWS) + 1j * rng.standard_normal(ROWS)
    bad = x.copy()
    bad[[17, 30000, 129999]] = [np.nan, np.inf, -np.inf + 1j * np.inf]
    want = {}
    try:
        tuning(b"spmv_skip_zero_blocks", 0)
        want = {k: spmv(plain, v) for k, v in (("x", x), ("bad", bad))}
    finally:
        tuning(b"spmv_skip_zero_blocks", 1)
    ref = O.spmv(M, O.spmv(M, x))
    assert np.max(np.abs(want["x"][0] + 1j * want["x"][1] - ref)) < 1e-12 * np.max(np.abs(ref))
    for rpt, C in got.items():
        for k in plain.diagonals[:: 29]:
            np.testing.assert_array_equal(np.asarray(C.get_diagonal(k)), np.asarray(plain.get_diagonal(k)))
        for k, v in (("x", x), ("bad", bad)):
            np.testing.assert_array_equal(spmv(C, v), want[k])
    C = got[0]
    ones = torch.ones(C.stored, dtype=torch.float64, device="cuda")
    zeros = torch.zeros_like(ones)
    capi.check(capi.lib().dq_devmat_set_packed_device(C.handle, ones.data_ptr(), zeros.data_ptr(), 0))
    torch.cuda.synchronize()
    E = O.Dia(ROWS, ROWS, list(C.diagonals), [np.ones(O.diagonal_length(o, ROWS, ROWS)) for o in C.diagonals])
    y = O.spmv(E, x)
    a, b = spmv(C, x)
    assert np.max(np.abs(a + 1j * b - y)) < 1e-12 * np.max(np.abs(y))


@pytest.mark.parametrize("zeros", [False, True])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("diags", [4, 16, 36])
def test_items_of_a_workgroup(diags, precision, zeros):
    """2^19 + 77 rows: 2 300, 25 000 and more than 65 536 items, one, two or four to a workgroup by their number and by how
    many blocks of the operands are zero; near diagonals with many pairs a result and far ones with few. The same values as
    without maps, where each workgroup has one."""
    import diaq_amd  # noqa: F401
    import diaq_gpu as d
    import torch
    from diaq_amd import capi
    rows = (1 << 19) + 77
    rng = np.random.default_rng(diags)
    for offs in (sorted(int(o) for o in rng.choice(np.arange(-rows // 2, rows // 2), diags, replace=False)),
                 list(range(-diags // 2, diags // 2))):
        vals = []
        for o in offs:
            n = rows - abs(o)
            v = rng.standard_normal(n) + 1j * rng.standard_normal(n)
            if zeros:
                v[(np.arange(n) + max(0, -o)) // 256 % 2 == 1] = 0
            vals.append(v)
        A = d.to_device(d.diaQMatrix.from_diagonals([rows, rows], offs, vals), precision)
        C = d.product(A, A)
        try:
            tuning(b"product_skip_zero_blocks", 0)
            plain = d.product(A, A)
        finally:
            tuning(b"product_skip_zero_blocks", 1)
        assert C.diagonals == plain.diagonals
        assert diags < 36 or offs[1] - offs[0] == 1 or len(C.diagonals) * (rows // 2048) > 1 << 16
        dt = torch.float64 if precision == "fp64" else torch.float32
        x = [torch.randn(rows, dtype=dt, device="cuda") for _ in range(2)]
        y = [[torch.empty_like(v) for v in x] for _ in range(2)]
        for M, (yr, yi) in zip((C, plain), y):
            capi.check(capi.lib().dq_spmv_device(M.handle, x[0].data_ptr(), x[1].data_ptr(), yr.data_ptr(), yi.data_ptr(), 0))
        torch.cuda.synchronize()
        assert torch.equal(y[0][0], y[1][0]) and torch.equal(y[0][1], y[1][1])
        for k in plain.diagonals[:: max(1, len(plain.diagonals) // 6)]:
            np.testing.assert_array_equal(np.asarray(C.get_diagonal(k)), np.asarray(plain.get_diagonal(k)))
        del C, plain


def test_a_large_result_keeps_its_map():
    """A result above 1 GiB with many zero blocks: its SpMV takes a NaN and infinities to the zeros as without the map, a
    sequence has its FP64 bits, and new values without zeros, and then with other zeros, are not read by the old map."""
    import diaq_amd  # noqa: F401
    import diaq_gpu as d
    import torch
    from diaq_amd import capi
    L = capi.lib()
    rows = (1 << 19) + 77
    rng = np.random.default_rng(11)
    offs = sorted(int(o) for o in rng.choice(np.arange(-rows // 2, rows // 2), 24, replace=False))
    vals = []
    for k, o in enumerate(offs):
        n = rows - abs(o)
        v = (rng.standard_normal(n) + (k % 2) * 1j * rng.standard_normal(n)) / 20
        v[(np.arange(n) + max(0, -o)) // (512 << k % 3) % 2 == 1] = 0
        vals.append(v)
    A = d.to_device(d.diaQMatrix.from_diagonals([rows, rows], offs, vals))
    C = d.product(A, A)
    assert 16 * C.stored > 1 << 30
    x = rng.standard_normal(rows) + 1j * rng.standard_normal(rows)
    bad = x.copy()
    bad[[17, 30000, 129999]] = [np.nan, np.inf, -np.inf + 1j * np.inf]

    def ntimes(M, v, n):
        t = [torch.as_tensor(p, device="cuda").contiguous() for p in (v.real, v.imag)]
        y, w = [torch.empty_like(p) for p in t], [torch.empty_like(p) for p in t]
        capi.check(L.dq_spmv_ntimes_device(M.handle, t[0].data_ptr(), t[1].data_ptr(), y[0].data_ptr(), y[1].data_ptr(), n,
                                           w[0].data_ptr(), w[1].data_ptr(), 0))
        torch.cuda.synchronize()
        return [p.cpu().numpy() for p in y]

    def compare(inputs):
        got = [(spmv(C, v), ntimes(C, x, 3)) for v in inputs]
        try:
            tuning(b"spmv_skip_zero_blocks", 0)
            want = [(spmv(C, v), ntimes(C, x, 3)) for v in inputs]
        finally:
            tuning(b"spmv_skip_zero_blocks", 1)
        for a, b in zip(got, want):
            np.testing.assert_array_equal(a, b)

    compare((x, bad))
    one = torch.ones(C.stored, dtype=torch.float64, device="cuda") / 1000
    for keep in (one > 0, torch.arange(C.stored, device="cuda") // 4096 % 2 == 0):
        re, im = one * keep, one * ~keep
        capi.check(L.dq_devmat_set_packed_device(C.handle, re.data_ptr(), im.data_ptr(), 0))
        torch.cuda.synchronize()
        compare((x, bad))
