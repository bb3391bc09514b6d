import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (gfx950) GPU and the built HIP library")


@pytest.fixture(autouse=True)
def automatic_gate_tiles():
    """Gate plans choose their tile for each test, whatever an earlier one left set: the tuning is the process's."""
    yield
    capi = sys.modules.get("diaq_amd.capi")
    if capi:
        for key in (b"gates_tile_qubits", b"gates_low_qubits"):
            capi.check(capi.lib().dq_set_tuning(key, 0))
