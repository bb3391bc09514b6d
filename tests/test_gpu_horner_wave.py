"""The wave form of the batched evolution's Horner level against a lane per state: the same bits with 1, 2, 4, 8 and 16
states, sizes that are no multiple of a wave, more than 64 diagonals, diagonals that end inside a wave, and blocks that are
zero in one part or both; and the values against a Taylor series in NumPy (FP32 values: 2e-6)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from oracle import oracle as O  # noqa: E402


def hamiltonian(rows, offs, seed):
    rng = np.random.default_rng(seed)
    vals = []
    for k, o in enumerate(offs):
        n = O.diagonal_length(o, rows, rows)
        r = np.arange(n) + max(0, -o)
        v = (rng.standard_normal(n) + 1j * rng.standard_normal(n)) / (2 * len(offs))
        v = (v, v.real + 0j, 1j * v.imag, v * (r // (16 << k % 4) % 2))[k % 4]
        vals.append(v.astype(np.complex64).astype(np.complex128))
    return O.Dia(rows, rows, list(offs), vals)


@pytest.mark.parametrize("n_states", [1, 2, 4, 8, 16])
@pytest.mark.parametrize("rows,reach", [(65, 2), (300, 40), (1025, 3), (4100, 9)])
def test_wave_form_has_the_same_bits(rows, reach, n_states):
    import diaq_amd  # noqa: F401
    import diaq_gpu as d
    from diaq_amd import capi, evolution
    L = capi.lib()
    offs = sorted({*range(-reach, reach + 1), -rows + 1, rows - 2, rows // 2})
    H = [hamiltonian(rows, offs, seed) for seed in (1, 2)]
    B = evolution.BatchedEvolution([d.to_device(d.diaQMatrix.from_diagonals([rows, rows], M.offsets, M.vals)) for M in H],
                                   n_states, "fp32")
    t, m, s = [0.9, 0.5], [7, 9], [1, 2]
    B.set_schedule(t, m, s)
    rng = np.random.default_rng(4)
    st = [rng.standard_normal((n_states, rows)) + 1j * rng.standard_normal((n_states, rows)) for _ in H]
    st = [v / np.linalg.norm(v, axis=1, keepdims=True) for v in st]

    def run(vec, rpt, du):
        for key, v in ((b"evo_vec", vec), (b"evo_rows_per_lane", rpt), (b"evo_diag_batch", du)):
            capi.check(L.dq_set_tuning(key, v))
        for j, v in enumerate(st):
            B.set_states(j, v)
        B.run(use_graph=False, renormalize=False)
        return [B.get_states(j, rows) for j in range(2)]

    try:
        base = run(0, 1, 0)
        for rpt, du in ((1, 1), (1, 2), (1, 4), (2, 2), (2, 4), (4, 0), (8, 0)):
            for a, b in zip(run(1, rpt, du), base):
                np.testing.assert_array_equal(a, b, err_msg=f"rpt={rpt} du={du}")
    finally:
        for key, v in ((b"evo_vec", -1), (b"evo_rows_per_lane", 0), (b"evo_diag_batch", 0)):
            capi.check(L.dq_set_tuning(key, v))
    for j, M in enumerate(H):
        for a, v in zip(base[j], st[j]):
            tau = t[j] / 2 ** s[j]
            for _ in range(2 ** s[j]):
                term = v
                for k in range(1, m[j] + 1):
                    term = O.spmv(M, term) * (-1j * tau / k)
                    v = v + term
            assert np.linalg.norm(a - v) < 2e-6


@pytest.mark.parametrize("precision", ["fp32", "fp64"])
@pytest.mark.parametrize("rows,diags,n_states", [(1, 1, 1), (63, 24, 8), (64, 7, 2), (1023, 24, 4), (1024, 23, 16),
                                                 (1024, 25, 8), (1025, 24, 1), (2048, 24, 8), (2049, 5, 1)])
def test_many_levels_in_one_launch(rows, diags, n_states, precision):
    """Small classes run all levels in one workgroup per state, up to 24 diagonals: the bits of a launch per level, also
    across launches (more than 4096 levels), for jobs of different lengths, and on replays of the graph."""
    import diaq_amd  # noqa: F401
    import diaq_gpu as d
    from diaq_amd import capi, evolution
    L = capi.lib()
    offs = sorted([0, *range(1, diags)], key=lambda k: (k * 7919) % 101)[:diags]
    offs = sorted({o if k % 2 else -o for k, o in enumerate(offs) if o < rows} | ({rows - 1} if rows > diags else set()))
    offs = offs[-diags:]
    H = [hamiltonian(rows, offs, seed) for seed in (1, 2)]
    B = evolution.BatchedEvolution([d.to_device(d.diaQMatrix.from_diagonals([rows, rows], M.offsets, M.vals)) for M in H],
                                   n_states, precision)
    B.set_schedule([0.7, 1.5], [7, 5], [3, 10])
    rng = np.random.default_rng(4)
    st = [rng.standard_normal((n_states, rows)) + 1j * rng.standard_normal((n_states, rows)) for _ in H]

    def run(vec, graph):
        capi.check(L.dq_set_tuning(b"evo_vec", vec))
        for j, v in enumerate(st):
            B.set_states(j, v)
        B.run(use_graph=graph, renormalize=True)
        return [B.get_states(j, rows) for j in range(2)]

    try:
        base = run(1, False)
        for graph in (False, True, True):
            for a, b in zip(run(-1, graph), base):
                np.testing.assert_array_equal(a, b)
    finally:
        capi.check(L.dq_set_tuning(b"evo_vec", -1))


@pytest.mark.parametrize("n_states", [1, 2, 16])
@pytest.mark.parametrize("rows", [1, 3, 257])
def test_states_cross_unchanged(rows, n_states):
    """Split and interleaved states in and out of a job: the same values back through either pair, per job."""
    import diaq_amd  # noqa: F401
    import diaq_gpu as d
    from diaq_amd import capi, evolution
    L = capi.lib()
    D = d.to_device(d.diaQMatrix.from_diagonals([rows, rows], [0], [np.ones(rows, complex)]))
    B = evolution.BatchedEvolution([D, D], n_states, "fp32")
    rng = np.random.default_rng(rows)
    st = [rng.standard_normal((n_states, rows)) + 1j * rng.standard_normal((n_states, rows)) for _ in range(2)]
    re, im = st[0].real.copy(), st[0].imag.copy()
    capi.check(L.dq_evo_set_states(B._h, 0, capi.ptr(re), capi.ptr(im)))
    B.set_states(1, st[1])
    for j in range(2):
        np.testing.assert_array_equal(B.get_states(j, rows), st[j])
        a, b = np.empty((n_states, rows)), np.empty((n_states, rows))
        capi.check(L.dq_evo_get_states(B._h, j, capi.ptr(a), capi.ptr(b)))
        np.testing.assert_array_equal(a + 1j * b, st[j])
    with pytest.raises(capi.DqError):
        capi.check(L.dq_evo_set_states_complex(B._h, 2, capi.ptr(st[0])))


@pytest.mark.parametrize("forced", [False, True])
@pytest.mark.parametrize("levels", [(1, 1), (1, 13), (11, 12), (12, 11), (13, 30)])
def test_lanes_of_few_kernels_beside_the_graph(levels, forced):
    """Two classes, of 2049 and 300 rows, with levels at both sides of what a graph takes (16 kernels: 12 levels and the
    norm), the small one also in the wave form (evo_vec = 1): on replays the bits of the launches without a graph, also after the levels of both have changed places."""
    import diaq_amd  # noqa: F401
    import diaq_gpu as d
    from diaq_amd import capi, evolution
    L = capi.lib()
    rows = (2049, 300)
    H = [hamiltonian(n, sorted({0, 1, -1, n // 3, -(n // 3)}), n) for n in rows]
    B = evolution.BatchedEvolution([d.to_device(d.diaQMatrix.from_diagonals([n, n], M.offsets, M.vals))
                                    for n, M in zip(rows, H)], 2, "fp32")
    assert B.n_classes == 2
    rng = np.random.default_rng(6)
    st = [rng.standard_normal((2, n)) + 1j * rng.standard_normal((2, n)) for n in rows]

    def run(graph):
        for j, v in enumerate(st):
            B.set_states(j, v)
        B.run(use_graph=graph, renormalize=True)
        return [B.get_states(j, n) for j, n in enumerate(rows)]

    try:
        capi.check(L.dq_set_tuning(b"evo_vec", 1 if forced else -1))
        for m in (levels, levels[::-1]):
            B.set_schedule([0.4, 0.7], m, [0, 0])
            base = run(False)
            for _ in range(3):
                for a, b in zip(run(True), base):
                    np.testing.assert_array_equal(a, b)
        for a, v, M, t, k in zip(base, st, H, (0.4, 0.7), m):
            for x, y in zip(a, v):
                term = want = y
                for i in range(1, k + 1):
                    term = O.spmv(M, term) * (-1j * t / i)
                    want = want + term
                assert np.linalg.norm(x - want / np.linalg.norm(want)) < 2e-6
    finally:
        capi.check(L.dq_set_tuning(b"evo_vec", -1))
