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
