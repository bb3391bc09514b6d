"""Gate plans with every kind of step at the automatic tile sizes (10, 11 and 12 tile qubits): layers of full one-qubit
gates, gates with few entries, full and sparse two-qubit gates, entries in descending slot order, runs of diagonal
gates on one to four qubits (in, across and outside the register window) and signed zeros. The same bits as the gates
one by one, zeros' signs included."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def unitary(rng, k):
    q, _ = np.linalg.qr(rng.standard_normal((k, k)) + 1j * rng.standard_normal((k, k)))
    return q


def gate(M, precision, keep=None, reverse=False):
    """M as a DeviceMatrix with its diagonals `keep` (all if None), in descending slot order if reverse."""
    import diaq_gpu as d
    n = M.shape[0]
    offs = sorted(range(-n + 1, n) if keep is None else keep, reverse=reverse)
    return d.to_device(d.diaQMatrix.from_diagonals([n, n], offs, [np.diagonal(M, o).copy() for o in offs]), precision)


def sequence(rng, n, precision):
    seq = [(gate(np.diag(np.exp(1j * rng.standard_normal(4))), precision, [0]), q) for q in range(n - 1)]
    seq += [(gate(unitary(rng, 2), precision), q) for q in range(n)]
    for q in rng.permutation(n - 3):
        q = int(q)
        kind = int(rng.integers(0, 9))
        if kind == 0:
            seq.append((gate(np.array([[0, 1], [1, 0]], complex), precision, [-1, 1]), q))
        elif kind == 1:
            seq.append((gate(unitary(rng, 4), precision), q))
        elif kind == 2:
            seq.append((gate(unitary(rng, 4), precision, [-1, 0, 1]), q))
        elif kind == 3:
            seq.append((gate(unitary(rng, 4), precision, reverse=True), q))
        elif kind == 4:
            seq.append((gate(unitary(rng, 2), precision, [0, 1], reverse=True), q))
        elif kind == 5:
            seq.append((gate(unitary(rng, 8), precision), q))
        else:
            k = kind - 5 + int(rng.integers(0, 2))
            seq.append((gate(np.diag(rng.choice([1, -1, 1j], 2 ** k)), precision, [0]), min(q, n - k)))
    return seq


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("n", [11, 12, 18, 19, 20, 21, 22])
def test_gate_windows_bitwise(n, precision):
    import diaq_amd  # noqa: F401
    import diaq_gpu as d
    import torch
    rng = np.random.default_rng(n)
    seq = sequence(rng, n, precision)
    plan = d.GatePlan(n, seq)
    dt = torch.float64 if precision == "fp64" else torch.float32
    g = torch.Generator(device="cuda").manual_seed(n)
    a = [torch.randn(1 << n, dtype=dt, device="cuda", generator=g) for _ in range(2)]
    for v in a:  # zeros of both signs in the state
        v[::7] = 0.0
        v[3::14] = -0.0
    b = [v.clone() for v in a]
    plan.run(a[0].data_ptr(), a[1].data_ptr(), repetitions=2)
    for _ in range(2):
        for G, q in seq:
            k = int(np.log2(G.shape[0]))
            d.kron_apply_device(G, n - q - k, q, b[0].data_ptr(), b[1].data_ptr(), b[0].data_ptr(), b[1].data_ptr(),
                                False)
    torch.cuda.synchronize()
    bits = torch.int64 if precision == "fp64" else torch.int32
    for v, w in zip(a, b):
        assert torch.equal(v.view(bits), w.view(bits))


def test_the_automatic_tile_comes_back():
    """0 sets both knobs back to automatic. A layer on 26 qubits: 12, 8 and 6 of them to a pass with 12-qubit tiles and four
    low qubits, which is the automatic choice; 11, 7, 7 and 1 with 11-qubit tiles; 12, 6, 6 and 2 with six low qubits."""
    import diaq_amd  # noqa: F401
    import diaq_gpu as d
    from diaq_amd import capi
    L = capi.lib()
    rng = np.random.default_rng(0)
    seq = [(gate(unitary(rng, 2), "fp64"), q) for q in range(26)]
    got = []
    for tile, low in ((0, 0), (11, 0), (0, 0), (0, 6), (0, 0)):
        capi.check(L.dq_set_tuning(b"gates_tile_qubits", tile))
        capi.check(L.dq_set_tuning(b"gates_low_qubits", low))
        got.append(d.GatePlan(26, seq).n_passes)
    assert got == [3, 4, 3, 4, 3]
