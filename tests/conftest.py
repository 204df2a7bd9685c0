import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs a real MI355X (run with -m gpu)")
    # the C-ABI library and the native calls are built in-tree beforehand; build them only if one is not there
    from actnn_amd import _lib
    if not (os.path.exists(_lib.LIB_PATH) and os.path.exists(_lib.HOST_PATH)):
        _lib.build()


@pytest.fixture(scope="session")
def lib():
    from actnn_amd import _lib
    return _lib.load()
