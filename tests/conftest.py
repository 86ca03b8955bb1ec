import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (runs through libdba_hip.so on cuda:0)")


def pytest_collection_modifyitems(items):
    # the folder of the reference's sources can be there and empty: what is built from them then has no sources
    ref = "/root/reference"
    if os.path.isdir(ref) and not os.listdir(ref):
        for item in items:
            if os.path.basename(str(item.fspath)) == "test_reference_tools.py":
                item.add_marker(pytest.mark.skip(reason="reference sources not present"))


@pytest.fixture(scope="session")
def ctx():
    from dba_amd import Context
    c = Context(0)
    yield c
    c.close()
