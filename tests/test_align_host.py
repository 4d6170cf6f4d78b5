"""Host side of the overlap aligner's batch (rh_align.cpp) on a stand-in for
the HIP runtime: what an error leaves behind, and how the slots share the
memory."""
import os
import subprocess

import pytest

from racon_amd import _lib

CSRC = os.path.join(_lib.PKG_DIR, "csrc")
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")


@pytest.fixture(scope="module")
def align_host(tmp_path_factory):
    exe = tmp_path_factory.mktemp("native") / "align_host"
    here = os.path.dirname(os.path.abspath(__file__))
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-D__HIP_PLATFORM_AMD__",
                    f"-I{ROCM}/include", f"-I{CSRC}/hip", f"-I{CSRC}/../../include", "-o", str(exe),
                    os.path.join(here, "native", "align_host.cpp"),
                    os.path.join(CSRC, "hip", "rh_align.cpp"), "-lpthread"],
                   check=True, capture_output=True)
    return str(exe)


@pytest.mark.parametrize("scenario", ["errors", "memory", "small"])
def test_batch(align_host, scenario):
    done = subprocess.run([align_host, scenario], capture_output=True, text=True, timeout=60)
    assert done.returncode == 0, done.stdout + done.stderr
