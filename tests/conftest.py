import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (gfx950) GPU")
    config.addinivalue_line("markers", "slow: long-running parity case")


@pytest.fixture(scope="session")
def orc():
    """The CPU oracle (test infrastructure), built on demand."""
    from oracle import oracle as O

    O.lib()
    return O


@pytest.fixture(scope="session")
def hip():
    """The HIP backend on device 0.  Fails (does not skip) if the library or
    the device is missing: GPU tests must run the native path."""
    import esolearn_amd as E

    E.init(0)
    info = E.HipBackend.device_info()
    print(f"[gpu] {info}", flush=True)
    return E


FAKE_PRELUDE = """
import ctypes as C, sys
import numpy as np
import esolearn_amd as E
F = C.CDLL(sys.argv[1])
F.fake_used.restype = C.c_size_t
F.fake_limit.argtypes = [C.c_size_t]
F.fake_launches.restype = F.fake_kernels.restype = C.c_char_p
def launches():
    return F.fake_launches().decode().splitlines()
E.init(0)
B = E.HipBackend
"""


@pytest.fixture(scope="session")
def fake_hip(tmp_path_factory):
    """Runs Python code in a fresh process on tests/fake_hip.cpp (a runtime
    without a device: host logic only, kernels are recorded and not run)."""
    lib = str(tmp_path_factory.mktemp("fake_hip") / "fake_hip.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-fPIC", "-shared",
                    os.path.join(ROOT, "tests", "fake_hip.cpp"), "-o", lib], check=True)

    def run(code):
        pre = " ".join(x for x in (lib, os.environ.get("LD_PRELOAD")) if x)
        r = subprocess.run([sys.executable, "-c", FAKE_PRELUDE + code, lib], capture_output=True, text=True, timeout=300,
                           cwd=ROOT, env={**os.environ, "LD_PRELOAD": pre})
        assert r.returncode == 0, r.stdout + r.stderr
        return r.stdout

    return run
