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
