"""Host copies by several threads, without a GPU: small ones start none, and a system without threads to give is no error."""
import subprocess
import sys
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
SHIM = ROOT / "tests" / "hipshim"


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    sys.path.insert(0, str(ROOT))
    from i_amd.build import ROCM

    out = tmp_path_factory.mktemp("copy") / "copy_threads"
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wno-unused-function", "-D__HIP_PLATFORM_AMD__", f"-I{ROCM / 'include'}", "-rdynamic",
                    str(SHIM / "copy_threads.cpp"), str(SHIM / "shim.cpp"), str(ROOT / "i_amd" / "csrc" / "runtime" / "host_copy.cpp"),
                    "-o", str(out), "-ldl", "-lpthread"], check=True)
    return out


@pytest.mark.parametrize("granted", [0, 1, 3, 20])
def test_threads_are_started_when_needed_and_may_be_refused(program, granted):
    done = subprocess.run([str(program), str(granted)], capture_output=True, text=True, timeout=100)
    assert done.returncode == 0, (done.stdout, done.stderr[-500:])
