import json
import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "pil2-proofman_amd")
for p in (ROOT, PKG):
    if p not in sys.path:
        sys.path.insert(0, p)

GOLDEN = os.path.join(ROOT, "tests", "golden")


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs a HIP GPU (MI355X); runs through libpil2_commit_hip.so")


def pytest_collection_modifyitems(items):
    """Tests that load the compiled reference come last. Where it is not built they fail,
    and a run that stops at the first failure (-x) would end before all others."""
    def loads_reference(item):
        code = [item.function] + [d[-1].func for d in item._fixtureinfo.name2fixturedefs.values()]
        return any("RefLib" in f.__code__.co_names for f in code if hasattr(f, "__code__"))

    items.sort(key=loads_reference)


@pytest.fixture(scope="session")
def oracle():
    from oracle.oracle import Oracle
    return Oracle()


@pytest.fixture(scope="session")
def refvec():
    with open(os.path.join(GOLDEN, "reference_vectors.json")) as f:
        return json.load(f)


@pytest.fixture(scope="session")
def compiled_ref():
    with open(os.path.join(GOLDEN, "compiled_reference.json")) as f:
        return json.load(f)


def hexes(lst):
    return [int(x, 16) for x in lst]
