"""The XPBD tile plan (spg_amd/csrc/xpbd_tiles.cpp) where memory runs out in one of its threads: the failure arrives at the
caller, who then steps group by group (tile_plan_memory.cpp)."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "spg_amd", "csrc")


def test_failed_allocations_arrive(tmp_path):
    exe = str(tmp_path / "check")
    subprocess.run(["g++", "-O2", "-std=c++17", "-pthread", f"-I{CSRC}", os.path.join(HERE, "tile_plan_memory.cpp"),
                    os.path.join(CSRC, "xpbd_tiles.cpp"), os.path.join(CSRC, "coloring.cpp"), "-o", exe], check=True)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0, out.stdout + out.stderr
