"""Zero-block maps of values with a few nonzeros to a block -- in its first rows, behind them, in its last row, in one part --
and the calls that skip by a map at sizes where one is made: the FP64 bits of the calls that read everything."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def lone_nonzeros(rows, seed, block=64):
    """Diagonals with one nonzero in some of their blocks, real, imaginary or both parts of it."""
    rng = np.random.default_rng(seed)
    offs = sorted({0, 1, -1, 5, -64, 77, 1000, -4099, rows // 2, -(rows // 2) + 3, rows - 9, -rows + 70})
    vals = []
    for k, o in enumerate(offs):
        r0, n = max(0, -o), rows - abs(o)
        v = np.zeros(n, complex)
        for b in range(r0 // block, (r0 + n - 1) // block + 1):
            at = block * b + (0, 7, 8, block // 2, block - 1)[int(rng.integers(0, 5))]
            if rng.random() < 0.7 and r0 <= at < r0 + n:
                v[at - r0] = (0.3, 0.2j, 0.1 - 0.4j)[(k + b) % 3]
        vals.append(v)
    return offs, vals


def tuned(key, value, call, back):
    from diaq_amd import capi
    try:
        capi.check(capi.lib().dq_set_tuning(key, value))
        return call()
    finally:
        capi.check(capi.lib().dq_set_tuning(key, back))


@pytest.mark.parametrize("rows", [1 << 16, (1 << 16) + 37])
def test_products_and_evolutions(rows):
    import diaq_amd  # noqa: F401
    import diaq_gpu as d
    import torch
    offs, vals = lone_nonzeros(rows, rows)
    A = d.to_device(d.diaQMatrix.from_diagonals([rows, rows], offs, vals))
    C, plain = d.product(A, A), tuned(b"product_skip_zero_blocks", 0, lambda: d.product(A, A), 1)
    assert C.diagonals == plain.diagonals
    for k in plain.diagonals:
        np.testing.assert_array_equal(np.asarray(C.get_diagonal(k)), np.asarray(plain.get_diagonal(k)))
    g = torch.Generator(device="cuda").manual_seed(rows)
    psi = [torch.randn(rows, dtype=torch.float64, device="cuda", generator=g) for _ in range(2)]

    def evolve():
        p = [v.clone() for v in psi]
        d.hamsim_device(A, p[0].data_ptr(), p[1].data_ptr(), 0.3, 2, 5)
        torch.cuda.synchronize()
        return p

    for a, b in zip(evolve(), tuned(b"hamsim_skip_zero_blocks", 0, evolve, 1)):
        assert torch.equal(a, b)


@pytest.mark.parametrize("n_states", [1, 2, 4, 8])
def test_batches(n_states):
    """The map's blocks are 256, 128, 64 and 32 rows here."""
    import diaq_amd  # noqa: F401
    import diaq_gpu as d
    from diaq_amd import evolution
    rows = 5003
    H = []
    for seed in (1, 2):
        offs, vals = lone_nonzeros(rows, seed, 256 // n_states)
        H.append(d.to_device(d.diaQMatrix.from_diagonals([rows, rows], offs, vals)))
    B = evolution.BatchedEvolution(H, n_states, "fp64")
    B.set_schedule([0.4, 0.7], [5, 6], [1, 0])
    rng = np.random.default_rng(n_states)
    st = [rng.standard_normal((n_states, rows)) + 1j * rng.standard_normal((n_states, rows)) for _ in H]

    def run():
        for j, v in enumerate(st):
            B.set_states(j, v)
        B.run(use_graph=False, renormalize=False)
        return [B.get_states(j, rows) for j in range(2)]

    for a, b in zip(run(), tuned(b"evo_skip_zero_blocks", 0, run, 1)):
        np.testing.assert_array_equal(a, b)


def hamiltonian(model, rows):
    """A TFIM or XXZ of 2^16 rows or more, or the first `rows` rows and columns of one."""
    from diaq_amd import hamiltonians as Hm
    q = int(np.ceil(np.log2(rows)))
    n, _, offs, vals = Hm.tfim(q, 1.0, 0.7) if model == "tfim" else Hm.xxz(q, seed=5)
    cut = [(o, np.asarray(v)[: rows - abs(o)]) for o, v in zip(offs, vals) if abs(o) < rows]
    return [o for o, _ in cut], [v for _, v in cut]


def state(rows, seed=3):
    rng = np.random.default_rng(seed)
    psi = rng.standard_normal(rows) + 1j * rng.standard_normal(rows)
    return psi / np.linalg.norm(psi)


@pytest.mark.parametrize("model", ["tfim", "xxz"])
@pytest.mark.parametrize("rows", [1 << 16, (1 << 16) + 4099])
def test_evolution_skips_exactly(model, rows):
    """From 2^16 rows on an evolution maps its matrix's zero blocks: FP64 the same bits as reading them, in every schedule of
    the terms; FP32 (compensated sums) within 5e-6, the bound of the smaller sizes' test."""
    import diaq_amd  # noqa: F401
    import diaq_gpu as d
    import torch
    from diaq_amd import capi
    from oracle import oracle as O
    L = capi.lib()
    offs, vals = hamiltonian(model, rows)
    psi, out = state(rows), {}
    try:
        for prec in ("fp64", "fp32"):
            D = d.to_device(d.diaQMatrix.from_diagonals([rows, rows], offs, vals), prec)
            dt = torch.float64 if prec == "fp64" else torch.float32
            for skip in (1, 0):
                for lds, rpt in ((0, 2), (1, 2), (-1, 0)):
                    capi.check(L.dq_set_tuning(b"hamsim_skip_zero_blocks", skip))
                    capi.check(L.dq_set_tuning(b"hamsim_lds", lds))
                    capi.check(L.dq_set_tuning(b"hamsim_rows_per_lane", rpt))
                    pr, pi = (torch.as_tensor(p, device="cuda").to(dt).contiguous() for p in (psi.real, psi.imag))
                    d.hamsim_device(D, pr.data_ptr(), pi.data_ptr(), 0.2, 2, 10)
                    torch.cuda.synchronize()
                    out[prec, skip, lds, rpt] = (pr.double() + 1j * pi.double()).cpu().numpy()
    finally:
        capi.check(L.dq_set_tuning(b"hamsim_skip_zero_blocks", 1))
        capi.check(L.dq_set_tuning(b"hamsim_lds", -1))
        capi.check(L.dq_set_tuning(b"hamsim_rows_per_lane", 0))
    base = out["fp64", 0, 0, 2]
    scale = np.max(np.abs(base))
    for key, v in out.items():
        if key[0] == "fp64":
            np.testing.assert_array_equal(v, base, err_msg=str(key))
        else:
            assert np.max(np.abs(v - base)) < 5e-6 * scale, key
    ref = O.hamiltonian_simulation(O.Dia(rows, rows, offs, vals), psi, 0.2, 2, 10)
    assert np.max(np.abs(base - ref)) < 1e-12 * np.max(np.abs(ref))


def ntimes(capi, entry, D, x, n, in_place=False, stream=0):
    import torch
    t = [torch.as_tensor(p, device="cuda").contiguous() for p in (x.real, x.imag)]
    w = [torch.empty_like(p) for p in t]
    y = t if in_place else [torch.empty_like(p) for p in t]
    capi.check(getattr(capi.lib(), entry)(D.handle, t[0].data_ptr(), t[1].data_ptr(), y[0].data_ptr(), y[1].data_ptr(), n,
                                          w[0].data_ptr(), w[1].data_ptr(), stream))
    torch.cuda.synchronize()
    return (y[0] + 1j * y[1]).cpu().numpy()


@pytest.mark.parametrize("model", ["tfim", "xxz"])
@pytest.mark.parametrize("rows", [1 << 16, (1 << 16) + 4099])
def test_sequences_skip_exactly(model, rows):
    """From 2^16 rows on spMV_ntimes maps an untuned matrix: FP64 the same bits with the skip on and off, in forced schedules,
    in place, from host vectors and tuned."""
    import diaq_amd  # noqa: F401
    import diaq_gpu as d
    from diaq_amd import capi
    from oracle import oracle as O
    L = capi.lib()
    offs, vals = hamiltonian(model, rows)
    H = d.diaQMatrix.from_diagonals([rows, rows], offs, vals)
    D, x, out = d.to_device(H), state(rows), {}
    try:
        for skip in (0, 1):
            capi.check(L.dq_set_tuning(b"spmv_skip_zero_blocks", skip))
            for lds, rpt in ((0, 1), (1, 4), (-1, 0)):
                capi.check(L.dq_set_tuning(b"spmv_lds", lds))
                capi.check(L.dq_set_tuning(b"spmv_rows_per_lane", rpt))
                for entry in ("dq_spmv_ntimes_device", "dq_spmv_ntimes_device_noalloc"):
                    for in_place in (False, True):
                        out[skip, lds, rpt, entry, in_place] = ntimes(capi, entry, D, x, 3, in_place)
            out[skip, "host"] = d.to_numpy_vector(d.spMV_ntimes(H, d.from_numpy_vector(x), 3))
        capi.check(L.dq_spmv_tune(D.handle, 2, 0, None))
        out["tuned"] = ntimes(capi, "dq_spmv_ntimes_device", D, x, 3)
    finally:
        capi.check(L.dq_set_tuning(b"spmv_skip_zero_blocks", 1))
        capi.check(L.dq_set_tuning(b"spmv_lds", -1))
        capi.check(L.dq_set_tuning(b"spmv_rows_per_lane", 0))
    base = out[0, -1, 0, "dq_spmv_ntimes_device", False]
    for key, v in out.items():
        np.testing.assert_array_equal(v, base, err_msg=str(key))
    ref = O.spmv_ntimes(O.Dia(rows, rows, offs, vals), x, 3)
    assert np.max(np.abs(base - ref)) < 1e-12 * np.max(np.abs(ref))


@pytest.mark.parametrize("in_place", [False, True])
def test_a_captured_sequence_maps_into_the_static_scratch(in_place):
    """The allocation-free sequence captured at a size that makes a map, replayed between eager calls of another matrix, also
    large enough, which write their maps over the same scratch."""
    import diaq_amd  # noqa: F401
    import diaq_gpu as d
    import torch
    from diaq_amd import capi
    rows, other = 1 << 17, (1 << 16) + 77
    D = d.to_device(d.diaQMatrix.from_diagonals([rows, rows], *hamiltonian("tfim", rows)))
    E = d.to_device(d.diaQMatrix.from_diagonals([other, other], *hamiltonian("xxz", other)))
    x, xo = state(rows), state(other, 4)
    want, want_other = (ntimes(capi, "dq_spmv_ntimes_device", M, v, 4) for M, v in ((D, x), (E, xo)))
    src = [torch.as_tensor(p, device="cuda").contiguous() for p in (x.real, x.imag)]
    t, w = [p.clone() for p in src], [torch.empty_like(p) for p in src]
    y = t if in_place else [torch.empty_like(p) for p in src]
    cs = torch.cuda.Stream()
    cs.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=cs):
        capi.check(capi.lib().dq_spmv_ntimes_device_noalloc(D.handle, t[0].data_ptr(), t[1].data_ptr(), y[0].data_ptr(),
                                                            y[1].data_ptr(), 4, w[0].data_ptr(), w[1].data_ptr(),
                                                            cs.cuda_stream))
    for _ in range(4):
        for p, q in zip(t, src):
            p.copy_(q)
        for p in w + ([] if in_place else y):
            p.fill_(7.0)
        np.testing.assert_array_equal(ntimes(capi, "dq_spmv_ntimes_device_noalloc", E, xo, 4), want_other)
        graph.replay()
        torch.cuda.synchronize()
        np.testing.assert_array_equal((y[0] + 1j * y[1]).cpu().numpy(), want)
