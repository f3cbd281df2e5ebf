"""The XPBD tile plan (spg_amd/csrc/xpbd_tiles.cpp) on the CPU: every particle goes through the same projections in the
same order as with one launch per group, and the plan's lists name only what they hold (tile_plan_check.cpp)."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "spg_amd", "csrc")


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("tiles") / "check")
    subprocess.run(["g++", "-O2", "-std=c++17", "-pthread", f"-I{CSRC}", os.path.join(HERE, "tile_plan_check.cpp"),
                    os.path.join(CSRC, "xpbd_tiles.cpp"), os.path.join(CSRC, "coloring.cpp"), "-o", exe], check=True)
    return exe


# tile edges (16 x 16 particles and one more), one tile, many; tiles whose needs do not fit (springs anywhere)
@pytest.mark.parametrize("kind,size", [("cloth", 2), ("cloth", 3), ("cloth", 16), ("cloth", 17), ("cloth", 33), ("cloth", 90),
                                       ("cloth", 150), ("cube", 1), ("cube", 6), ("cube", 14), ("net", 40), ("net", 9000)])
@pytest.mark.parametrize("serial", [0, 1])
@pytest.mark.parametrize("threads", [512, 1024])
def test_plan_equals_one_launch_per_group(check, kind, size, serial, threads):
    if serial and size > 100 and kind == "cloth":
        pytest.skip("thousands of levels: the same code as smaller cloths")
    out = subprocess.run([check, kind, str(size), str(serial), str(threads)], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout
    if kind != "net" and size > 2:
        assert not out.stdout.startswith("batches 0"), out.stdout


# one launch takes as long as its workgroups follow each other on a compute unit: 256 tiles at a time on 256 of them
@pytest.mark.parametrize("kind,size,threads,tiled", [("cloth", 512, 1024, True), ("cloth", 1024, 1024, True), ("cube", 17, 512, True),
                                                     ("cube", 48, 512, True), ("cube", 64, 512, False)])
def test_tiles_where_they_are_faster(check, kind, size, threads, tiled):
    """Measured, a substep in tiles and with a launch per group, us: cloths 33 and 84, 125 and 182; solids 60 and 91, 84 and
    128, and 221 and 152 where 64^3 cells are cut into 538 tiles."""
    out = subprocess.run([check, kind, str(size), "0", str(threads)], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout
    assert (int(out.stdout.split()[3]) > 0) == tiled, out.stdout
