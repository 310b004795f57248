import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X GPU and the built HIP library")


def gpu_available():
    try:
        import torch
        return torch.cuda.is_available()
    except Exception:
        return False


@pytest.fixture(scope="session")
def engine():
    if not gpu_available():
        pytest.skip("no GPU")
    from phinfortran_amd import transport
    eng = transport.Engine(0)
    yield eng
    eng.close()


@pytest.fixture(params=[True, False], ids=["planes", "layers"])
def both_paths(engine, request):
    """Run a test twice: with batched solves on the planes of the principal
    layers where the blocks have them (the default), and on whole layers, whose
    mixed-precision, split and shared-lead paths the planes would bypass."""
    engine.set_planes(request.param)
    yield request.param
    engine.set_planes(True)
