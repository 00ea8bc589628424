import gc
import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs a real MI355X (run with -m gpu)")


@pytest.fixture(scope="module", autouse=True)
def no_garbage_of_earlier_files():
    """networks of one file that wait for the collector (modules in cycles, up to 200 MB on the device) are gone before the next file
    begins: tests that compare what the device holds before and after a call would see them go in between"""
    gc.collect()


@pytest.fixture(scope="session")
def oracle():
    import oracle as orc
    return orc
