"""What bench.py says about a tile, for every tile there is."""
import re
import shutil
import subprocess
import sys

import pytest

import amrhip
from conftest import ROOT

sys.path.insert(0, ROOT)
import bench  # noqa: E402


@pytest.mark.parametrize("n", [2, 4, 8, 16])
def test_every_tile_has_a_design_text(n):
    tiles = amrhip.tile_variants(n)
    assert tiles and all(bench.DESIGNS[design] for _, _, design in tiles)


@pytest.mark.skipif(shutil.which("nm") is None, reason="nm absent")
@pytest.mark.parametrize("n", [2, 4, 8, 16])
def test_the_kernel_named_is_one_of_the_library(n):
    """`name<args, ...>` begins the name of a kernel that the library holds"""
    out = subprocess.run(["nm", "-C", amrhip.LIB_PATH], capture_output=True, text=True, check=True).stdout
    held = set(re.findall(r"stage_kernel\w*<[^>]*>", out))
    assert held
    for tile in amrhip.tile_variants(n):
        name = bench.kernel_name(n, tile)
        begin = name[:-len("...>")] if name.endswith("...>") else name
        assert any(k.startswith(begin) for k in held), name
    line = bench.roofline_of(1000, 1.0, 10, n, amrhip.tile_variants(n)[-1], "direct stream launches", [0.1] * 3)
    assert line["kernel"] == bench.kernel_name(n, amrhip.tile_variants(n)[-1])


@pytest.mark.parametrize("workload,cells", [("batch64", 6924352), ("riemann4", 207424), ("vortex_l9_n8", 16777216)])
def test_counted_traffic_is_of_the_kernel_that_runs(workload, cells):
    """the committed counters are those of the default tile's kernel, and are
    not given for another kernel or mesh"""
    name = bench.kernel_name(8, (1, 5, 1))
    traffic, tile = bench.measured_traffic(workload, cells, name)
    assert tile == "1,5,1" and 1.0 < traffic / (cells * bench.B_ALG_STAGE) < 1.1
    assert bench.measured_traffic(workload, cells, bench.kernel_name(8, (1, 4, 1))) == (traffic, tile)
    assert bench.measured_traffic(workload, cells, "stage_kernel<8, 1, 5, 1, ...>") is None
    assert bench.measured_traffic(workload, cells + 64, name) is None
