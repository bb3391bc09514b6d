"""Evolution of matrices that fit one workgroup, at the sizes around its limits (rows a wave, a workgroup, two rows per lane
in FP32; 1 to 24 diagonals, and one more) against a Taylor series in NumPy. FP64: 1e-12. FP32 values: the terms round to
FP32, the state does not, so the error stays below 8 eps32 = 1e-6 for ||H|| t of order one."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from oracle import oracle as O  # noqa: E402

CASES = [(1, 1), (2, 3), (63, 24), (64, 7), (65, 23), (700, 24), (1000, 25), (1023, 13), (1024, 24), (1024, 1), (1025, 5),
         (1999, 21), (2048, 24), (2049, 9)]


def hamiltonian(rows, diags, dtype):
    rng = np.random.default_rng(rows + diags)
    half = (diags - 1) // 2
    near = [o for o in (1, 2, 3, 5, 8, 16, 31, 64, 100, 255, 256, 300) if o < rows][:half]
    if half and rows > 4:
        near[-1] = min(rows - 1, 511)
    offs = sorted({0, *near, *(-o for o in near)})
    if diags % 2 == 0 and rows > 6:
        offs.append(4)
    vals = []
    for o in offs:
        n = O.diagonal_length(o, rows, rows)
        v = (rng.standard_normal(n) + 1j * rng.standard_normal(n)) / (2 * len(offs))
        vals.append(v.astype(dtype).astype(np.complex128))
    return O.Dia(rows, rows, sorted(offs), [v for _, v in sorted(zip(offs, vals), key=lambda p: p[0])])


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("case", CASES)
def test_small_evolution(case, precision):
    import diaq_amd  # noqa: F401
    import diaq_gpu as d
    import torch
    rows, diags = case
    H = hamiltonian(rows, diags, np.complex64 if precision == "fp32" else np.complex128)
    D = d.to_device(d.diaQMatrix.from_diagonals([rows, rows], H.offsets, H.vals), precision)
    rng = np.random.default_rng(3)
    psi = rng.standard_normal(rows) + 1j * rng.standard_normal(rows)
    psi /= np.linalg.norm(psi)
    steps, m, dt = 3, 9, 0.21
    want = psi
    for _ in range(steps):
        term = want
        for k in range(1, m + 1):
            term = O.spmv(H, term) * (-1j * dt / k)
            want = want + term
    if precision == "fp32":  # the FP32 form ends with the norm it started with
        want = want / np.linalg.norm(want)
    pr, pi = (torch.as_tensor(p, device="cuda").contiguous() for p in (psi.real, psi.imag))
    d.hamsim_device_fp64_state(D, pr.data_ptr(), pi.data_ptr(), dt * steps, steps, m, 0)
    torch.cuda.synchronize()
    got = (pr + 1j * pi).cpu().numpy()
    assert np.linalg.norm(got - want) < (1e-12 if precision == "fp64" else 1e-6)


@pytest.mark.parametrize("key,value", [(b"hamsim_lds", 0), (b"hamsim_rows_per_lane", 2), (b"hamsim_skip_zero_blocks", 0)])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("case", [(1, 1), (65, 23), (1000, 24), (1024, 13), (1999, 21), (2048, 24)])
def test_an_override_asks_for_a_launch_per_term(case, precision, key, value):
    """The terms' own schedule, which each override selects, and one workgroup for all of them: the same bits, also where the
    steps take several launches (more than 4096 terms)."""
    import diaq_amd  # noqa: F401
    import diaq_gpu as d
    import torch
    from diaq_amd import capi
    rows, diags = case
    H = hamiltonian(rows, diags, np.complex64 if precision == "fp32" else np.complex128)
    D = d.to_device(d.diaQMatrix.from_diagonals([rows, rows], H.offsets, H.vals), precision)
    rng = np.random.default_rng(5)
    psi = rng.standard_normal(rows) + 1j * rng.standard_normal(rows)
    L, off = capi.lib(), {b"hamsim_lds": -1, b"hamsim_rows_per_lane": 0, b"hamsim_skip_zero_blocks": 1}[key]
    out = []
    for steps, m in ((2, 7), (600, 7)):
        for v in (off, value):
            pr, pi = (torch.as_tensor(p, device="cuda").contiguous() for p in (psi.real, psi.imag))
            try:
                capi.check(L.dq_set_tuning(key, v))
                d.hamsim_device_fp64_state(D, pr.data_ptr(), pi.data_ptr(), 0.01 * steps, steps, m, 0)
            finally:
                capi.check(L.dq_set_tuning(key, off))
            torch.cuda.synchronize()
            out.append((pr.cpu().numpy(), pi.cpu().numpy()))
        np.testing.assert_array_equal(out[-1], out[-2])
