import os
import sys

import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs a ROCm GPU (MI355X); run with -m gpu")


def _has_gpu() -> bool:
    try:
        return torch.cuda.is_available()
    except Exception:
        return False


def pytest_collection_modifyitems(config, items):
    if _has_gpu():
        return
    skip = pytest.mark.skip(reason="no GPU in this environment")
    for it in items:
        if "gpu" in it.keywords:
            it.add_marker(skip)


@pytest.fixture(scope="session")
def dev():
    return torch.device("cuda:0")


@pytest.fixture(scope="session")
def shim_lib(tmp_path_factory):
    import ctypes
    import subprocess

    from kernel_collections_amd import _lib
    so = str(tmp_path_factory.mktemp("shim") / "liblaunch_shim.so")
    subprocess.check_call(["g++", "-O1", "-shared", "-fPIC", "-o", so, os.path.join(ROOT, "tests", "launch_shim.cpp"), "-ldl"])
    lib = ctypes.CDLL(so)
    assert lib.shim_init(_lib.LIB_PATH.encode()) == 0
    return so, lib


@pytest.fixture
def shim(shim_lib):
    """The native host layer over launch_shim.cpp: yields the shim, whose counters tell what a call did."""
    import ctypes

    from kernel_collections_amd import _lib
    so, lib = shim_lib
    lib.count = lambda name: ctypes.c_int.in_dll(lib, name).value
    native = _lib.native()
    for name in ("shim_launches", "shim_stage1", "shim_locked_calls", "shim_poison", "shim_poisoned"):
        ctypes.c_int.in_dll(lib, name).value = 0
    native.init(so)
    try:
        yield lib
    finally:
        native.init(_lib.LIB_PATH)
