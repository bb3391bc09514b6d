"""Several products with a band matrix in one launch against a launch per product: the same bits at sizes around a
workgroup's 512 rows, for 1 to 40 diagonals (and one more), uneven bands, odd counts, x == y, and a NaN and an infinity in x;
and the oracle's values (1e-12 in FP64, 2e-6 in FP32)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from oracle import oracle as O  # noqa: E402

BANDS = {"one": [0], "tri": [-1, 0, 1], "up": [1, 2, 7], "wide": list(range(-16, 17)), "full": list(range(-25, 15)),
         "more": list(range(-20, 21)), "gaps": [-60, -3, 0, 40]}


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("band", BANDS)
@pytest.mark.parametrize("rows", [1, 63, 512, 513, 1500, 70001])
def test_band_powers(rows, band, precision):
    import diaq_amd  # noqa: F401
    import diaq_gpu as d
    import torch
    from diaq_amd import capi
    L = capi.lib()
    offs = [o for o in BANDS[band] if -rows < o < rows]
    if not offs:
        pytest.skip("the band has no diagonal at this size")
    rng = np.random.default_rng(rows)
    vals = []
    for o in offs:
        n = O.diagonal_length(o, rows, rows)
        vals.append((rng.standard_normal(n) + 1j * rng.standard_normal(n)) / np.sqrt(2 * len(offs)))
    M = O.Dia(rows, rows, offs, vals)
    D = d.to_device(d.diaQMatrix.from_diagonals([rows, rows], offs, vals), precision)
    dt = torch.float64 if precision == "fp64" else torch.float32
    x = rng.standard_normal(rows) + 1j * rng.standard_normal(rows)
    bad = x.copy()
    bad[rows // 3] = np.nan
    bad[-1] = np.inf

    def run(v, n, in_place=False):
        xr, xi = (torch.as_tensor(p, device="cuda").to(dt).contiguous() for p in (v.real, v.imag))
        yr, yi = (xr, xi) if in_place else (torch.full_like(xr, 7.0), torch.full_like(xr, 7.0))
        wr, wi = torch.full_like(xr, 5.0), torch.full_like(xr, 5.0)
        capi.check(L.dq_spmv_ntimes_device(D.handle, xr.data_ptr(), xi.data_ptr(), yr.data_ptr(), yi.data_ptr(), n,
                                           wr.data_ptr(), wi.data_ptr(), 0))
        torch.cuda.synchronize()
        return np.stack([yr.cpu().numpy(), yi.cpu().numpy()])

    cases = [(x, 2), (x, 4), (x, 5), (x, 11), (bad, 3)]
    got = [run(v, n) for v, n in cases]
    placed = [run(v, n, True) for v, n in cases]
    try:
        capi.check(L.dq_set_tuning(b"spmv_xcd", 0))  # a launch per product
        want = [run(v, n) for v, n in cases]
    finally:
        capi.check(L.dq_set_tuning(b"spmv_xcd", -1))
    for a, b, w in zip(got, placed, want):
        np.testing.assert_array_equal(a, w)
        np.testing.assert_array_equal(b, w)
    ref = x
    for _ in range(4):
        ref = O.spmv(M, ref)
    err = np.max(np.abs(got[1][0] + 1j * got[1][1] - ref))
    assert err <= (1e-12 if precision == "fp64" else 2e-6) * max(np.max(np.abs(ref)), 1e-30)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("n", [3, 5, 7, 9, 11, 15])
def test_x_as_the_work_vector(n, precision):
    """An odd count needs x for its first product only, so x may also be the work vector, however many launches it takes."""
    import diaq_amd  # noqa: F401
    import diaq_gpu as d
    import torch
    from diaq_amd import capi
    L = capi.lib()
    rows = 200003
    rng = np.random.default_rng(n)
    for band in ("tri", "wide", "gaps"):
        offs = BANDS[band]
        vals = [rng.standard_normal(rows - abs(o)) / len(offs) + 0j for o in offs]
        D = d.to_device(d.diaQMatrix.from_diagonals([rows, rows], offs, vals), precision)
        dt = torch.float64 if precision == "fp64" else torch.float32
        x = rng.standard_normal((2, rows))
        out = []
        for shared in (False, True):
            xr, xi = (torch.as_tensor(p, device="cuda").to(dt).contiguous() for p in x)
            yr, yi = torch.empty_like(xr), torch.empty_like(xi)
            wr, wi = (xr, xi) if shared else (torch.empty_like(xr), torch.empty_like(xi))
            capi.check(L.dq_spmv_ntimes_device(D.handle, xr.data_ptr(), xi.data_ptr(), yr.data_ptr(), yi.data_ptr(), n,
                                               wr.data_ptr(), wi.data_ptr(), 0))
            torch.cuda.synchronize()
            out.append((yr.cpu().numpy(), yi.cpu().numpy()))
        np.testing.assert_array_equal(out[0], out[1], err_msg=band)
