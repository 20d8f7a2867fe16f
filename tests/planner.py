"""The library's planner on the CPU: csrc/runtime.cpp built against
tests/planner_stub.cpp instead of HIP, and the Python package loaded on top of it
under another name.  Calls plan and "launch" as on a GPU; `launched()` tells what
they would have run."""

import ctypes
import importlib.util
import os
import subprocess
import sys
import tempfile
from functools import lru_cache
from pathlib import Path

ROOT = Path(__file__).resolve().parents[1]
PACKAGE = ROOT / "triton-metal_amd"
ROCM = Path(os.environ.get("ROCM_PATH", "/opt/rocm"))


def buildable() -> bool:
    return (PACKAGE / "lib" / "blobs.S").exists() and (ROCM / "include").exists()


@lru_cache(maxsize=None)
def _library() -> str:
    out = Path(tempfile.mkdtemp(prefix="tm_planner_")) / "libplanner.so"
    subprocess.run(
        ["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__",
         f"-I{ROCM / 'include'}", f"-I{PACKAGE / 'csrc'}", str(PACKAGE / "csrc" / "runtime.cpp"),
         str(PACKAGE / "csrc" / "codeobject.cpp"), str(ROOT / "tests" / "planner_stub.cpp"),
         str(PACKAGE / "lib" / "blobs.S"), "-o", str(out), f"-L{ROCM / 'lib'}", "-lhiprtc",
         f"-Wl,-rpath,{ROCM / 'lib'}", "-Wl,-Bsymbolic"], check=True)
    return str(out)


@lru_cache(maxsize=None)
def package():
    """(ops, DeviceBuffer) of the triton_metal package over the stub library."""
    name = "triton_metal_planner"
    directory = PACKAGE / "triton_metal"
    saved = os.environ.get("TRITON_METAL_CORE_LIB")
    os.environ["TRITON_METAL_CORE_LIB"] = _library()
    try:
        spec = importlib.util.spec_from_file_location(
            name, directory / "__init__.py", submodule_search_locations=[str(directory)])
        sys.modules[name] = importlib.util.module_from_spec(spec)
        spec.loader.exec_module(sys.modules[name])
        ops = importlib.import_module(name + ".ops")
        buffer = importlib.import_module(name + ".buffer")
    finally:
        if saved is None:
            del os.environ["TRITON_METAL_CORE_LIB"]
        else:
            os.environ["TRITON_METAL_CORE_LIB"] = saved
    return ops, buffer.DeviceBuffer


def launched():
    """(name, (gx, gy, gz), threads, dynamic LDS) of every launch since the last call."""
    lib = ctypes.CDLL(_library())
    text = ctypes.create_string_buffer(1 << 16)
    assert lib.planner_take_log(text, len(text)) >= 0
    rows = [line.split() for line in text.value.decode().splitlines()]
    return [(r[0], tuple(map(int, r[1:4])), int(r[4]), int(r[5])) for r in rows]
