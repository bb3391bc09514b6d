"""Gate plans on states with infinities, NaNs and amplitudes that overflow inside a pass: what the gates one by one give (NaN
where they give NaN). In FP32 a compensated row sum whose first term is infinite is NaN, one whose last term is stays infinite."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

N = 13


def gate(M, precision, keep=None, reverse=False):
    import diaq_gpu as d
    n = M.shape[0]
    offs = sorted(range(-n + 1, n) if keep is None else keep, reverse=reverse)
    return d.to_device(d.diaQMatrix.from_diagonals([n, n], offs, [np.diagonal(M, o).copy() for o in offs]), precision)


def unitary(rng, k):
    q, _ = np.linalg.qr(rng.standard_normal((k, k)) + 1j * rng.standard_normal((k, k)))
    return q


def cross(t, s=1.0):
    return s * np.array([[np.cos(t), -1j * np.sin(t)], [-1j * np.sin(t), np.cos(t)]])


def sequences(rng, precision, tile):
    one = [(unitary(rng, 2), {}), (unitary(rng, 2), dict(reverse=True)), (unitary(rng, 4), {}),
           (unitary(rng, 4), dict(reverse=True)), (unitary(rng, 2), dict(keep=[0, 1])), (unitary(rng, 4), dict(keep=[-1, 0, 2])),
           (np.diag(np.exp(1j * rng.standard_normal(4))), dict(keep=[0]))]
    for M, how in one:
        for q in (0, 4, 9, N - 2):
            yield [(gate(M, precision, **how), q)]
    for s in (1.0, 3.0, 40.0):  # one layer
        yield [(gate(cross(rng.uniform(0.6, 0.9), s), precision), q) for q in range(5, 5 + tile - 8)]
    for s in (1.0, 5.0, 40.0):  # layers of rotations about X, and scaled ones that overflow sooner
        yield [(gate(cross(rng.uniform(0.2, 1.3), s), precision), q) for q in range(N)]
    yield [(gate(cross(1e-3 if q else 1.4), precision), q) for q in range(N)]
    yield [(gate(unitary(rng, 2), precision), q) for q in range(N)]
    yield [(gate(10 * unitary(rng, 2), precision, reverse=q % 2 == 1), q) for q in range(N)]


@pytest.mark.parametrize("tile", [10, 11, 12])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_extreme_amplitudes(precision, tile):
    import diaq_amd  # noqa: F401
    import diaq_gpu as d
    import torch
    from diaq_amd import capi
    rng = np.random.default_rng(tile)
    real = np.float64 if precision == "fp64" else np.float32
    dt = torch.float64 if precision == "fp64" else torch.float32
    big = float(np.finfo(real).max)
    base = rng.standard_normal((2, 1 << N))
    states = {"finite": base}
    states["infinite"] = base.copy()
    states["infinite"][0, [3, 700]] = np.inf, -np.inf
    states["infinite"][1, [5001]] = np.inf
    states["nan"] = base.copy()
    states["nan"][1, [17, 4099]] = np.nan
    states["near the largest"] = rng.uniform(0.4, 0.7, (2, 1 << N)) * big * rng.choice([-1, 1], (2, 1 << N))
    states["one large"] = base.copy()
    states["one large"][0, 129] = 0.9 * big
    states["one large"][1, 130] = -0.9 * big
    capi.check(capi.lib().dq_set_tuning(b"gates_tile_qubits", tile))
    for i, seq in enumerate(sequences(rng, precision, tile)):
        plan = d.GatePlan(N, seq)
        for name, st in states.items():
            a = [torch.as_tensor(v.astype(real), device="cuda").contiguous() for v in st]
            b = [v.clone() for v in a]
            plan.run(a[0].data_ptr(), a[1].data_ptr(), repetitions=1)
            for G, q in seq:
                k = int(np.log2(G.shape[0]))
                d.kron_apply_device(G, N - q - k, q, b[0].data_ptr(), b[1].data_ptr(), b[0].data_ptr(), b[1].data_ptr(),
                                    False)
            torch.cuda.synchronize()
            for v, w in zip(a, b):
                np.testing.assert_array_equal(v.cpu().numpy(), w.cpu().numpy(), err_msg=f"sequence {i}, {name}")
