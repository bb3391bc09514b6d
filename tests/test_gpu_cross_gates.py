"""Layers of gates with real diagonal and imaginary other entries inside a pass: the bits of the gates one by one, with finite
states and with a NaN and infinities among the amplitudes, at each tile size; and layers that hold one general gate."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("tile", [10, 11, 12])
@pytest.mark.parametrize("general", [False, True])
def test_cross_layers(tile, precision, general):
    import diaq_amd  # noqa: F401
    import diaq_gpu as d
    import torch
    from diaq_amd import capi
    n = 15
    rng = np.random.default_rng(n)

    def gate(m):
        return d.to_device(d.diaQMatrix.from_diagonals([2, 2], [-1, 0, 1], [np.array([m[1, 0]]), np.diag(m).copy(),
                                                                            np.array([m[0, 1]])]), precision)

    gates = []
    for q in range(n):
        t = rng.uniform(0.1, 1.4)
        m = np.array([[np.cos(t), -1j * np.sin(t)], [-0.7j * np.sin(t), 0.9 * np.cos(t)]])
        if general and q % 6 == 1:
            m = m + 0.3 * (1 + 1j)
        gates.append((gate(m), q))
    dt = torch.float64 if precision == "fp64" else torch.float32
    psi = rng.standard_normal(1 << n) + 1j * rng.standard_normal(1 << n)
    bad = psi.copy()
    bad[[5, 4097, 30000]] = [np.nan, np.inf, 2 - 1j * np.inf]
    try:
        capi.check(capi.lib().dq_set_tuning(b"gates_tile_qubits", tile))
        plan = d.GatePlan(n, gates)
    finally:
        capi.check(capi.lib().dq_set_tuning(b"gates_tile_qubits", 11))
    for state in (psi, bad):
        ar, ai, br, bi = (torch.as_tensor(p, device="cuda").to(dt).contiguous()
                          for p in (state.real, state.imag, state.real, state.imag))
        plan.run(ar.data_ptr(), ai.data_ptr(), 1, 0)
        for G, q in gates:
            d.kron_apply_device(G, n - q - 1, q, br.data_ptr(), bi.data_ptr(), br.data_ptr(), bi.data_ptr(), False)
        torch.cuda.synchronize()
        np.testing.assert_array_equal(ar.cpu().numpy(), br.cpu().numpy())
        np.testing.assert_array_equal(ai.cpu().numpy(), bi.cpu().numpy())
