"""The proof service's scheduling on the CPU: service.hip compiled as host code over
stand-ins of the prover core (service_standins.cpp)."""
import ctypes
import shutil
import subprocess

import pytest

from sqd import build

pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")


@pytest.fixture(scope="module")
def service(tmp_path_factory):
    lib = tmp_path_factory.mktemp("service") / "service.so"
    cmd = ["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-pthread", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include"]
    cmd += build._inc() + ["-x", "c++", str(build.PKG / "csrc" / "service.hip"),
                           str(build.ROOT / "tests" / "service_standins.cpp"), "-o", str(lib)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-4000:]
    lib = ctypes.CDLL(str(lib))
    lib.service_waits.restype = ctypes.c_long
    return lib


@pytest.mark.parametrize("workers", [2, 3, 8])
def test_workers_waiting_for_memory_sleep(service, workers):
    # one program holds the only core for 0.3 s while the workers of the others wait
    # for its memory.  A worker sleeps a few times per job (its wake-ups for a job,
    # a core and a freed row, each of which may wake all others): at most some
    # 10 * workers^2 waits.  Workers that wake each other give 1e4 and more.
    waits = service.service_waits(workers, 300)
    assert 0 <= waits <= 10 * workers * workers + 100
