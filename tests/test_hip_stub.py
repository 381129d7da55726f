"""The library's host code over a stub of the HIP runtime (no GPU): what it
allocates and frees, and what a failed call leaves behind.  The scenarios are
in ``hip_stub_driver.c``."""

from __future__ import annotations

import gc
import shutil
import subprocess
import types
import weakref
from pathlib import Path

import pytest
import torch

from seoulkv_amd import SeoulKV4, _hip
from seoulkv_amd.ref_runtime import GroupOutput
from seoulkv_amd.result import DecodeResult

HERE = Path(__file__).resolve().parent


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    if shutil.which("gcc") is None:
        pytest.skip("gcc not installed")
    exe = tmp_path_factory.mktemp("stub") / "hip_stub_driver"
    lib = _hip.LIB_PATH
    subprocess.run(["gcc", "-std=gnu11", "-O1", "-g", "-Wall", "-Wextra", "-Werror",
                    "-D__HIP_PLATFORM_AMD__", "-isystem", "/opt/rocm/include",
                    "-I", str(HERE.parent / "include"), str(HERE / "hip_stub_driver.c"),
                    "-o", str(exe), "-rdynamic", "-L", str(lib.parent), "-lseoulkv4_hip",
                    f"-Wl,-rpath,{lib.parent}"], check=True)
    return exe


@pytest.mark.parametrize("scenario", ["output_lifetime", "failed_run"])
def test_host_code_over_the_stub_runtime(driver, scenario):
    res = subprocess.run([str(driver), scenario], capture_output=True, text=True, timeout=120)
    assert res.returncode == 0, (res.returncode, res.stdout, res.stderr)
    assert f"hip stub driver ok: {scenario}" in res.stdout


class _Lib:
    """Stands for the library: notes when a handle and its outputs are freed."""

    def __init__(self):
        self.events = []

    def skv_output_hold(self, handle, hold):
        hold._obj.value = 0x77
        return 0

    def skv_output_release(self, hold):
        self.events.append("outputs")

    def skv_destroy(self, handle):
        self.events.append("caches")

    def skv_sync(self, handle, status):
        return 0

    def skv_output_tiles_device(self, handle, ptr):
        ptr._obj.value = 0x1000
        return 0


class _Pages:
    """Stands for a page pool, whose device memory goes with the object."""


def _instance(lib):
    runtime = _hip.Runtime.__new__(_hip.Runtime)
    runtime.lib, runtime.handle, runtime.device = lib, 0x55, 0
    runtime._pool = _Pages()
    runtime.output = _hip.OutputMemory(lib, runtime.handle)
    attn = SeoulKV4.__new__(SeoulKV4)
    attn._state, attn._closed, attn._generation, attn._device = runtime, False, 1, 0
    attn._kv_pool = attn._pages = attn._host_kv = attn._index = attn._status = None
    return attn


@pytest.fixture
def views(monkeypatch):
    """torch.as_tensor over a device pointer keeps the wrapper it is given, as
    the real tensor does; nothing reads the pointer."""
    class View:
        def __init__(self, wrapper, device):
            self.wrapper = wrapper

        def view(self, dtype):
            return self

        def __getitem__(self, g):
            return self

    monkeypatch.setattr(torch, "as_tensor", View)


@pytest.mark.parametrize("how", ["close", "drop"])
def test_output_view_keeps_the_outputs_and_nothing_else(views, how):
    lib = _Lib()
    attn = _instance(lib)
    pages = weakref.ref(attn._state._pool)
    view = DecodeResult(attn, 1).device_tensors
    if how == "close":
        attn.close()
    del attn
    gc.collect()
    assert lib.events == ["caches"]  # freed under the live view, the outputs not
    assert pages() is None
    del view
    gc.collect()
    assert lib.events == ["caches", "outputs"]


def test_group_output_view_keeps_the_outputs_and_nothing_else(views):
    lib = _Lib()
    attn = _instance(lib)
    runtime, attn._state = attn._state, None
    view = GroupOutput(runtime, 2).device_view()
    alive = weakref.ref(runtime)
    runtime.close()
    assert lib.events == ["caches"]
    del runtime
    gc.collect()
    assert alive() is None and lib.events == ["caches"]
    del view
    gc.collect()
    assert lib.events == ["caches", "outputs"]


def test_instance_without_views_frees_all():
    for close in (True, False):
        lib = _Lib()
        attn = _instance(lib)
        if close:
            attn.close()
        del attn
        gc.collect()
        assert lib.events == ["caches", "outputs"]


def test_instance_that_never_initialised_drops_quietly():
    attn = SeoulKV4.__new__(SeoulKV4)
    del attn
    attn = _instance(types.SimpleNamespace(skv_output_hold=lambda h, p: 0,
                                           skv_output_release=lambda p: None))
    attn._state = None
    del attn
    gc.collect()
