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
