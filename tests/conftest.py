"""Test configuration: the `gpu` marker, import paths and shared fixtures."""
import os
import sys

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(REPO, "tpds22-artifact_amd")
for p in (PKG, os.path.join(REPO, "tests")):
    if p not in sys.path:
        sys.path.insert(0, p)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (runs the HIP kernels)")


# Files whose tests have to come before the others of the process, whatever they are
# called: cooperative launches of this process can make those of the command-line
# programs, run as its children, fail; and a launch whose stream shares one of HIP's four
# hardware queues with a running serving loop waits for the loop, so loops run while the
# process has few streams.
FIRST = ["test_gpu_cli.py", "test_gpu_serve.py", "test_gpu_fullsize.py"]


def pytest_collection_modifyitems(items):
    items.sort(key=lambda i: FIRST.index(i.path.name) if i.path.name in FIRST else len(FIRST))


@pytest.fixture(scope="session")
def oracle():
    import oracle_lib
    return oracle_lib.load()


@pytest.fixture(scope="session")
def hs():
    import hsync
    hsync.load()
    return hsync


@pytest.fixture(scope="session")
def arena(hs):
    a = hs.Arena()
    yield a
    a.close()
