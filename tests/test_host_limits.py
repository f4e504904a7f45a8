"""Host code where memory runs out (CPU, no GPU)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CS = os.path.join(ROOT, "gpu4hophl_code_amd", "csrc")
ROCM = "/opt/rocm"


@pytest.mark.slow
def test_staging_is_returned_without_memory(tmp_path):
    """The staging pool takes a call's staging back in a destructor: with no
    memory to be had it may not throw, since that would end the caller's
    process (tests/stage_driver.cpp)."""
    hipcc = os.path.join(ROCM, "bin", "hipcc")
    if not os.path.exists(hipcc) or not shutil.which("g++"):
        pytest.skip("compilers not installed")
    inc = ["-I", os.path.join(ROOT, "include"), "-I", CS]
    objs = []
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-fPIC", "-pthread", *inc, "-c",
                           os.path.join(CS, "graph.cpp"), "-o", str(tmp_path / "graph.o")])
    objs.append(str(tmp_path / "graph.o"))
    for src in (os.path.join(CS, "index.hip"), os.path.join(CS, "parents.hip"),
                os.path.join(ROOT, "tests", "stage_driver.cpp")):
        obj = str(tmp_path / (os.path.basename(src) + ".o"))
        subprocess.check_call([hipcc, "-x", "hip", "--offload-arch=gfx950", "-O1", "-std=c++17",
                               "-fPIC", *inc, "-Xclang", "-target-feature", "-Xclang",
                               "-packed-fp32-ops", "-c", src, "-o", obj],
                              stderr=subprocess.DEVNULL)
        objs.append(obj)
    exe = str(tmp_path / "drv")
    subprocess.check_call([hipcc, "--offload-arch=gfx950", *objs, "-o", exe, "-lpthread"])
    out = subprocess.run([exe], capture_output=True, text=True, timeout=120,
                         env=dict(os.environ, HIP_VISIBLE_DEVICES=""))
    assert out.returncode == 0, (out.returncode, out.stdout, out.stderr[-2000:])
    assert "stages returned" in out.stdout
