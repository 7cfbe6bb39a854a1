"""Host side of the GPU re-layout without a GPU (tests/hostsim/relayout_growth.cpp):
after an allocation failed, no kernel is given memory that is not there."""
import os
import pathlib
import subprocess

ROOT = pathlib.Path(__file__).resolve().parent.parent


def test_workspace_after_a_failed_allocation(tmp_path):
    src = ROOT / "tests" / "hostsim" / "relayout_growth.cpp"
    obj, exe = tmp_path / "relayout_growth.o", tmp_path / "relayout_growth"
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    subprocess.run([hipcc, "-x", "hip", "--offload-host-only", "-O1", "-fPIC", "-std=c++17",
                    "-I", str(ROOT / "include"), "-I", str(ROOT / "yoxel-voxel_amd" / "csrc"), "-c", str(src),
                    "-o", str(obj)], check=True)
    subprocess.run(["g++", str(obj), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
