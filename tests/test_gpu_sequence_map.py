"""The map that the first product of a sequence leaves for the others, at its edges: one or two rows per lane, more than 64
diagonals, a last block with few rows, diagonals that end inside a block, zeros in one part, both or neither. FP64: the bits of
products that read everything; both precisions, and both device entry points, against the oracle (1e-12, 2e-6)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from oracle import oracle as O  # noqa: E402


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("rows", [1 << 16, (1 << 16) + 1, (1 << 18) + 65])
@pytest.mark.parametrize("near", [3, 40])
def test_first_product_leaves_the_map(rows, near, precision):
    import diaq_amd  # noqa: F401
    import diaq_gpu as d
    import torch
    from diaq_amd import capi
    L = capi.lib()
    rng = np.random.default_rng(rows + near)
    offs = sorted({*range(-near, near + 1), 700, -4096, rows // 2 + 3, rows - 30, -rows + 70})
    vals = []
    for k, o in enumerate(offs):
        n = O.diagonal_length(o, rows, rows)
        r = np.arange(n) + max(0, -o)
        v = (rng.standard_normal(n) + 1j * rng.standard_normal(n)) / np.sqrt(2 * len(offs))
        v = (v, v.real + 0j, 1j * v.imag, v * (r // 64 % 2), v * (r // 192 % 2), 0 * v)[k % 6]
        vals.append(v)
    M = O.Dia(rows, rows, offs, vals)
    D = d.to_device(d.diaQMatrix.from_diagonals([rows, rows], offs, vals), precision)
    x = rng.standard_normal(rows) + 1j * rng.standard_normal(rows)
    dt = torch.float64 if precision == "fp64" else torch.float32
    ref = O.spmv(M, O.spmv(M, O.spmv(M, x)))

    def run(entry):
        xr, xi = (torch.as_tensor(p, device="cuda").to(dt).contiguous() for p in (x.real, x.imag))
        yr, yi, wr, wi = (torch.full_like(xr, 3.0) for _ in range(4))
        capi.check(getattr(L, entry)(D.handle, xr.data_ptr(), xi.data_ptr(), yr.data_ptr(), yi.data_ptr(), 3,
                                     wr.data_ptr(), wi.data_ptr(), 0))
        torch.cuda.synchronize()
        return (yr.double() + 1j * yi.double()).cpu().numpy()

    got = run("dq_spmv_ntimes_device")
    np.testing.assert_array_equal(run("dq_spmv_ntimes_device_noalloc"), got)
    assert np.max(np.abs(got - ref)) < (1e-12 if precision == "fp64" else 2e-6) * np.max(np.abs(ref))
    if precision == "fp64":
        try:
            capi.check(L.dq_set_tuning(b"spmv_skip_zero_blocks", 0))
            np.testing.assert_array_equal(run("dq_spmv_ntimes_device"), got)
        finally:
            capi.check(L.dq_set_tuning(b"spmv_skip_zero_blocks", 1))
