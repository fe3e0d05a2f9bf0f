"""CPU: eigenvectors of a dense batch that nobody took over are freed with it,
as when a solve ends with an error between the batch and its use."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_untaken_vectors_are_freed(tmp_path):
    exe = str(tmp_path / "drv")
    r = subprocess.run(["g++", "-std=c++17", "-O0", "-D__HIP_PLATFORM_AMD__", f"-I{ROCM}/include",
                        os.path.join(HERE, "dense_batch_driver.cpp"), "-o", exe], capture_output=True, text=True,
                       timeout=200)
    assert r.returncode == 0, r.stderr[-3000:]
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr[-2000:]
