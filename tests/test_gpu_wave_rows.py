"""The wave form of the row kernels (64 or 128 rows per wave, diagonals in ballots of 64) at the sizes where it can go
wrong, against the oracle: rows around a wave and a workgroup, more than 64 diagonals, diagonals that start or end
inside a wave, rectangular shapes, two rows per lane (from 2^18 rows) with odd tails, and zero-block maps with blocks
whose real part, imaginary part or both are zero. Tolerances as the other SpMV tests: 1e-12 in FP64, 2e-6 in FP32."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from oracle import oracle as O  # noqa: E402


def rel(a, b):
    return float(np.max(np.abs(a - b)) / np.max(np.abs(b)))


def matrix(rows, cols, offs, seed, scale=1.0):
    rng = np.random.default_rng(seed)
    vals = []
    for k, o in enumerate(offs):
        n = O.diagonal_length(o, rows, cols)
        v = scale * (rng.standard_normal(n) + 1j * rng.standard_normal(n))
        r = np.arange(n) + max(0, -o)  # the row of each value
        if k % 4 == 1:
            v = v.real + 0j
        elif k % 4 == 2:
            v = 1j * v.imag
        elif k % 4 == 3:
            v = v * (r // (64 << (k % 3)) % 2)
        vals.append(v)
    return O.Dia(rows, cols, list(offs), vals)


def device(M, precision):
    import diaq_gpu as d
    return d.to_device(d.diaQMatrix.from_diagonals([M.rows, M.cols], M.offsets, M.vals), precision)


def vectors(x, dt):
    import torch
    return [torch.as_tensor(p, device="cuda").to(dt).contiguous() for p in (x.real, x.imag)]


SHAPES = [(1, 1), (63, 63), (64, 65), (65, 64), (129, 200), (257, 257), (1000, 700), ((1 << 18) + 1, 1 << 18),
          ((1 << 18) + 129, (1 << 18) + 300)]


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("shape", SHAPES)
def test_wave_form_spmv_edges(shape, precision):
    import diaq_amd  # noqa: F401
    import diaq_gpu as d
    import torch
    rows, cols = shape
    near = [o for o in range(-37, 38) if -rows < o < cols]
    far = [-rows + 1, -rows + 3, -(rows // 2) - 5, rows // 3, cols - 2, cols - 1]
    M = matrix(rows, cols, sorted({o for o in near + far if -rows < o < cols}), rows)
    rng = np.random.default_rng(1)
    x = rng.standard_normal(cols) + 1j * rng.standard_normal(cols)
    dt = torch.float64 if precision == "fp64" else torch.float32
    xr, xi = vectors(x, dt)
    yr, yi = (torch.full((rows,), float("nan"), dtype=dt, device="cuda") for _ in range(2))
    d.spmv_device(device(M, precision), xr.data_ptr(), xi.data_ptr(), yr.data_ptr(), yi.data_ptr(), 0)
    torch.cuda.synchronize()
    got = (yr.double() + 1j * yi.double()).cpu().numpy()
    assert rel(got, O.spmv(M, x)) < (1e-12 if precision == "fp64" else 2e-6)


@pytest.mark.parametrize("entry", ["dq_spmv_ntimes_device", "dq_spmv_ntimes_device_noalloc"])
@pytest.mark.parametrize("rows", [1 << 16, (1 << 16) + 77, (1 << 18) + 33])
def test_wave_form_skips_zero_blocks_and_parts(rows, entry):
    """Two products with the map of 64-row blocks (both entry points): the oracle's values, and in FP64 the same bits as
    reading every block; FP32 within its bound."""
    import diaq_amd  # noqa: F401
    import torch
    from diaq_amd import capi
    L = capi.lib()
    M = matrix(rows, rows, sorted([-rows + 40, -4097, -300, -64, -1, 0, 1, 2, 63, 64, 129, 5000, rows - 70]), 7, 0.3)
    rng = np.random.default_rng(2)
    x = rng.standard_normal(rows) + 1j * rng.standard_normal(rows)
    ref = O.spmv(M, O.spmv(M, x))

    def run(D, dt):
        xr, xi = vectors(x, dt)
        yr, yi, wr, wi = (torch.empty_like(xr) for _ in range(4))
        capi.check(getattr(L, entry)(D.handle, xr.data_ptr(), xi.data_ptr(), yr.data_ptr(), yi.data_ptr(), 2,
                                     wr.data_ptr(), wi.data_ptr(), 0))
        torch.cuda.synchronize()
        return (yr.double() + 1j * yi.double()).cpu().numpy()

    D = device(M, "fp64")
    got = run(D, torch.float64)
    try:
        capi.check(L.dq_set_tuning(b"spmv_skip_zero_blocks", 0))
        np.testing.assert_array_equal(got, run(D, torch.float64))
    finally:
        capi.check(L.dq_set_tuning(b"spmv_skip_zero_blocks", 1))
    assert rel(got, ref) < 1e-12
    assert rel(run(device(M, "fp32"), torch.float32), ref) < 2e-6
