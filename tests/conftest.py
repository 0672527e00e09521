import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
for p in (os.path.join(ROOT, "tests"), os.path.join(ROOT, "md-lab_amd"), ROOT):
    if p not in sys.path:
        sys.path.insert(0, p)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (HIP device) to run")


@pytest.fixture(scope="session")
def golden():
    from orc import read_golden
    return read_golden()


@pytest.fixture(scope="session")
def oracle():
    from orc import Oracle
    return Oracle()


@pytest.fixture(autouse=True)
def engine_settings(request):
    """The engine's settings are process-wide; a GPU test leaves the chain length
    as it was and the Ewald parameters as a fresh process has them, so that no
    test measures what another one set."""
    if request.node.get_closest_marker("gpu") is None:
        yield
        return
    import pyxmd
    lib = pyxmd.Lib()
    M = lib.md_get_nhc_length_x()
    yield
    lib.md_set_nhc_length_x(M)
    lib.md_set_coulomb_truc_x(0.0)
    lib.md_set_coulomb_n_sum_x(0)
    lib.md_set_ewald_split_x(-1.0)
