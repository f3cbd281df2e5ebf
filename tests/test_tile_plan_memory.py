"""The XPBD tile plan (spg_amd/csrc/xpbd_tiles.cpp) where memory runs out in one of its threads: the failure arrives at the
caller, who then steps group by group (tile_plan_memory.cpp); no other error is taken for one (memory_errors.cpp)."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "spg_amd", "csrc")
INCLUDE = os.path.join(os.path.dirname(HERE), "include")


def test_failed_allocations_arrive(tmp_path):
    exe = str(tmp_path / "check")
    subprocess.run(["g++", "-O2", "-std=c++17", "-pthread", f"-I{CSRC}", os.path.join(HERE, "tile_plan_memory.cpp"),
                    os.path.join(CSRC, "xpbd_tiles.cpp"), os.path.join(CSRC, "coloring.cpp"), "-o", exe], check=True)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0, out.stdout + out.stderr


def test_only_memory_errors_are_done_without(tmp_path):
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    exe = str(tmp_path / "errors")
    subprocess.run(["g++", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", f"-I{CSRC}", f"-I{INCLUDE}", f"-I{rocm}/include",
                    os.path.join(HERE, "memory_errors.cpp"), "-o", exe, f"-L{rocm}/lib", f"-Wl,-rpath,{rocm}/lib",
                    "-lamdhip64"], check=True)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0, out.stdout + out.stderr
