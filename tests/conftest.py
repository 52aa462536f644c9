import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)
sys.path.insert(0, os.path.join(ROOT, "oracle"))


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (runs through libmilc_hip.so on cuda:0)")
    config.addinivalue_line("markers", "slow: longer CPU oracle checks")


@pytest.fixture(params=[1, 0], ids=["small-lattice-form", "large-lattice-form"])
def small_form(request):
    """Both forms of the solves on a small lattice, for Lattice.set_small_lattice_form:
    a lattice that the oracle solves quickly takes the one-kernel solves (1); the
    launch-by-launch and batched ones of larger lattices are tested on it too (0)."""
    return request.param


@pytest.fixture(scope="session")
def oracle():
    import ks_oracle
    return ks_oracle
