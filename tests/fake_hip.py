"""Tests of the library's host code on a HIP runtime without a device (native/fake_hip.cpp).

A test module runs one of its functions with `isolated`: in a process of its own, where the
fake runtime is loaded with global symbols before libpbrtm.so. There `install` sets the hooks."""
import ctypes
import os
import shutil
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROCM = "/opt/rocm/include"
needs_compiler = pytest.mark.skipif(shutil.which("g++") is None or not os.path.isdir(ROCM), reason="needs g++ and ROCm's headers")

_LAUNCH = ctypes.CFUNCTYPE(ctypes.c_int, ctypes.c_char_p, ctypes.c_uint32, ctypes.c_uint32, ctypes.c_int,
                           ctypes.POINTER(ctypes.c_void_p))
_GRAPH = ctypes.CFUNCTYPE(ctypes.c_int)
_OCCUPANCY = ctypes.CFUNCTYPE(ctypes.c_int, ctypes.c_char_p)
_keep = []


def isolated(module_file, function, tmp_path, *args, timeout=120):
    """Runs function(*args) (strings) of the module in a new process; fails with its output."""
    lib = tmp_path / "fake_hip.so"
    subprocess.run(["g++", "-std=c++17", "-O1", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__", f"-I{ROCM}", "-o",
                    str(lib), os.path.join(HERE, "native", "fake_hip.cpp")], check=True)
    env = dict(os.environ, PBRTM_FAKE_HIP=str(lib))
    p = subprocess.run([sys.executable, module_file, function, *args], capture_output=True, text=True, env=env,
                       timeout=timeout)
    assert p.returncode == 0, f"exit code {p.returncode}\n{p.stdout[-2000:]}\n{p.stderr[-4000:]}"


def main(namespace):
    """The new process's entry point: `if __name__ == "__main__": fake_hip.main(globals())`."""
    namespace[sys.argv[1]](*sys.argv[2:])


def install(launch=None, graph=None, occupancy=None):
    """launch(kernel, blocks, threads, captured, args) and graph() return an error code or None;
    occupancy(kernel) the resident workgroups per compute unit. Returns the fake runtime."""
    lib = ctypes.CDLL(os.environ["PBRTM_FAKE_HIP"], mode=ctypes.RTLD_GLOBAL)
    hooks = (_LAUNCH(lambda k, b, t, c, a: (launch(k.decode(), b, t, bool(c), a) if launch else 0) or 0),
             _GRAPH(lambda: (graph() if graph else 0) or 0),
             _OCCUPANCY(lambda k: occupancy(k.decode()) if occupancy else 1))
    _keep.append(hooks)
    lib.fake_hip_hooks(*hooks)
    return lib


def pointer(args, k):
    """Kernel argument k as an address."""
    return ctypes.cast(args[k], ctypes.POINTER(ctypes.c_uint64)).contents.value


def poke_u32(address, value):
    ctypes.c_uint32.from_address(address).value = value
