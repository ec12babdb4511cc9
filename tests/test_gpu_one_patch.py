"""The one-patch stage kernel of the 8x8 tiles where its edge round is least
regular: sides with a wall, one neighbour and two fine neighbours on one patch,
patches that are their own neighbours, stopped instances."""
import numpy as np
import pytest

import amrhip
from test_gpu_rows import small_forest

pytestmark = pytest.mark.gpu


def results(tile, scheme, insts, arrays):
    g = amrhip.Gpu()
    g.setup(8, scheme, insts, *arrays[:4], arrays[4])
    g.set_tile(*tile)
    got = [g.rhs()]
    norm = g.run(3)
    got += [g.soln(), *g.time()]
    g.close()
    return got, norm


@pytest.mark.parametrize("scheme", [1, 2, 3, 4, 5])
def test_mixed_edges_equal_the_other_tiles(scheme):
    """a single periodic patch, a single patch between walls, random adaptive
    forests with and without walls, one instance stopped after its first step:
    residual, states, times and step sizes are bit for bit those of a two-patch
    tile, whose edge faces come from a task list"""
    forests = [small_forest(8, 11, True, 0, 0), small_forest(8, 12, False, 0, 0), small_forest(8, 13, False, 1, 4),
               small_forest(8, 14, True, 1, 4), small_forest(8, 15, False, 2, 3)]
    bcs = [(0, 0, 0, 0), (1, 2, 0, 1), (2, 1, 1, 0), (0, 0, 0, 0), (0, 1, 2, 1)]
    insts = [amrhip.make_inst(1.0, bc, 0.2, 1e-3 * (1 + k), 1e-9 if k == 2 else 0.0) for k, bc in enumerate(bcs)]
    arrays = amrhip.batch_external(forests)
    ref, ref_norm = results((2, 4, 1), scheme, insts, arrays)
    for tile in [t for t in amrhip.tile_variants(8) if t[0] == 1]:
        got, norm = results(tile, scheme, insts, arrays)
        for a, b in zip(got, ref):
            assert np.array_equal(a, b), tile
        # the norm sums each tile's workgroups in its own order
        assert abs(norm - ref_norm) <= 1e-12 * ref_norm
