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


def _build_shim(folder, name):
    import ctypes
    import subprocess

    from kernel_collections_amd import _lib
    so = str(folder / f"lib{name}.so")
    subprocess.check_call(["g++", "-O1", "-shared", "-fPIC", "-o", so, os.path.join(ROOT, "tests", name + ".cpp"), "-ldl"])
    lib = ctypes.CDLL(so)
    assert lib.shim_init(_lib.LIB_PATH.encode()) == 0
    return so, lib


def _over_shim(so, lib):
    import ctypes

    from kernel_collections_amd import _lib
    lib.count = lambda name: ctypes.c_int.in_dll(lib, name).value
    native = _lib.native()
    for name in ("shim_launches", "shim_stage1", "shim_locked_calls", "shim_poison", "shim_poisoned"):
        ctypes.c_int.in_dll(lib, name).value = 0
    native.init(so)
    try:
        yield lib
    finally:
        native.init(_lib.LIB_PATH)


@pytest.fixture(scope="session")
def shim_lib(tmp_path_factory):
    return _build_shim(tmp_path_factory.mktemp("shim"), "launch_shim")


@pytest.fixture(scope="session")
def shim_tail_lib(tmp_path_factory):
    return _build_shim(tmp_path_factory.mktemp("shim"), "launch_shim_tail")


@pytest.fixture
def shim(shim_lib):
    """The native host layer over launch_shim.cpp: yields the shim, whose counters tell what a call did.  It has the entry points of the ABI version,
    not those added to it since."""
    yield from _over_shim(*shim_lib)


@pytest.fixture
def shim_tail(shim_tail_lib):
    """The same over launch_shim_tail.cpp, which has them."""
    yield from _over_shim(*shim_tail_lib)
