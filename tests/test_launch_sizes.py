"""Launches of a stage on the CPU: the launch code itself, built for the host with
a launch macro that records (tests/launch_sizes.cpp).

The runtime takes fewer than 2^32 threads along an axis of a launch and at most
65535 blocks along y and z.  Routed sweeps fill each plane's lines up to whole
tiles, so thin grids that fit the device have more tiles than one launch of
256-thread blocks may: the grids below need 2^24 and more.  Every tile of every
axis is computed once, however the blocks are divided into launches.

Which plain FP64 grids take k_sweep_split: both sides of the rule, which the GPU
test of the same grids runs.
"""
import shutil
import subprocess
from pathlib import Path

import pytest

from test_gpu_sweep_paths import SPLIT_EDGE

ROOT = Path(__file__).resolve().parents[1]
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"

pytestmark = pytest.mark.skipif(not Path(HIPCC).exists(), reason="hipcc not found")


@pytest.fixture(scope="module")
def stage_launches(tmp_path_factory):
    """stage_launches(n, bc, form) -> ([(kernel, grid, block, first block)], {axis: (tiles, once, more)})"""
    exe = {}
    for exact in (0, 1):
        exe[exact] = tmp_path_factory.mktemp("launches") / f"launch_sizes{exact}"
        cmd = [HIPCC, "-std=c++17", "-O1", "--offload-host-only", f"-DHOWMHD_EXACT={exact}", f"-I{ROOT / 'include'}",
               f"-I{ROOT / 'how-mhd-kokkos_amd' / 'csrc'}", str(ROOT / "tests" / "launch_sizes.cpp"), "-o", str(exe[exact])]
        build = subprocess.run(cmd, capture_output=True, text=True, timeout=300)
        assert build.returncode == 0, build.stderr[-3000:]

    def run(n, bc, form):
        arg = ",".join(map(str, (*n, int(bc == "open"), form)))
        r = subprocess.run([str(exe[0 if form.startswith("fp32") else 1]), arg], capture_output=True, text=True, timeout=120)
        assert r.returncode == 0, r.stdout + r.stderr
        launches, tiles = [], {}
        for line in r.stdout.splitlines():
            w = line.split()
            if w[0] == "launch":
                launches.append((w[1], tuple(map(int, w[2:5])), int(w[5]), int(w[6])))
            elif w[0] == "tiles":
                tiles[w[1]] = tuple(map(int, w[2:]))
        return launches, tiles

    return run


@pytest.mark.parametrize("n,bc,form", [((1, 8192, 8192), "periodic", "fp32i"), ((1, 8192, 8192), "open", "fp64i"),
                                       ((4, 6000, 6000), "open", "fp32i"), ((3, 7000, 7000), "periodic", "fp32i"),
                                       ((1, 16384, 16384), "open", "fp32i"), ((512, 512, 512), "open", "fp64"),
                                       ((97, 75, 61), "open", "fp32i"), ((97, 120, 130), "periodic", "fp64"),
                                       ((32, 32, 32), "periodic", "fp64"), ((128, 128, 1), "open", "fp64"),
                                       ((2000001, 1, 1), "open", "fp64"), ((3, 5, 65535), "open", "fp64i")])
def test_launches_fit_and_cover(n, bc, form, stage_launches):
    launches, tiles = stage_launches(n, bc, form)
    for kernel, grid, block, _ in launches:
        assert grid[0] * block < 2 ** 32, (kernel, grid)
        assert all(g <= 65535 for g in grid[1:]), (kernel, grid)
    for axis, (want, once, more) in tiles.items():
        assert (once, more) == (want, 0), axis
    assert {a for a, t in tiles.items() if t[0]} == {a for a, k in zip("xyz", n) if k > 1}


@pytest.mark.parametrize("n,bc,split", SPLIT_EDGE + [((128, 128, 1), "open", False), ((800, 1, 1), "open", True),
                                                     ((256, 256, 256), "periodic", False)])
def test_split_sides(n, bc, split, stage_launches):
    launches, _ = stage_launches(n, bc, "fp64")
    assert any("k_sweep_split" in kernel for kernel, *_ in launches) == split
    assert any("k_sweep<" in kernel for kernel, *_ in launches) != split
