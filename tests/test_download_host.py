"""download() built for the CPU against a stand-in for the HIP runtime
(tests/native): what cannot be brought about on a device."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CXX = shutil.which("g++")


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    if CXX is None:
        pytest.skip("no host compiler")
    out = str(tmp_path_factory.mktemp("native") / "download_host")
    native = os.path.join(HERE, "native")
    csrc = os.path.join(ROOT, "microsimulator_amd", "csrc")
    subprocess.run([CXX, "-std=c++20", "-O1", "-w", "-pthread", f"-I{native}", f"-I{csrc}",
                    f"-I{os.path.join(ROOT, 'include')}",
                    os.path.join(native, "download_host.cpp"),
                    os.path.join(csrc, "download.cpp"), "-o", out], check=True)
    return out


@pytest.mark.parametrize("what", ["registered", "allocations"])
def test_download(program, what):
    done = subprocess.run([program, what], capture_output=True, text=True, timeout=120)
    assert done.returncode == 0, done.stdout + done.stderr
