import os
import sys

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(REPO, "quasi-linear-kernel-attention_amd")
for p in (REPO, PKG):
    if p not in sys.path:
        sys.path.insert(0, p)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an AMD GPU (MI355X) and the built libqlka.so")


def _gpu_available():
    try:
        import torch
        return torch.cuda.is_available()
    except Exception:  # noqa: BLE001
        return False


def pytest_collection_modifyitems(config, items):
    if _gpu_available():
        return
    skip = pytest.mark.skip(reason="no GPU visible")
    for it in items:
        if "gpu" in it.keywords:
            it.add_marker(skip)


@pytest.fixture(scope="session")
def dev():
    import torch
    return torch.device("cuda", 0)


# The library's own routing by size ("auto"), or every short segment too through sort + walk or, where N + M allows it,
# sort + column sums: dense cutoff (None: as it is), column mode.
ROUTES = {"auto": (None, 0), "walk": (0, 1), "columns": (0, 2)}


@pytest.fixture
def pin_route():
    """pin_route(name) routes the library's calls as ROUTES says until the test ends."""
    from qlka import _lib
    lib = _lib.load()
    cutoff, mode = lib.qlka_set_direct_max(512), lib.qlka_set_columns(0)
    lib.qlka_set_direct_max(cutoff)

    def pin(name):
        direct_max, columns = ROUTES[name]
        lib.qlka_set_direct_max(cutoff if direct_max is None else direct_max)
        lib.qlka_set_columns(columns)
        return name

    yield pin
    lib.qlka_set_direct_max(cutoff)
    lib.qlka_set_columns(mode)
