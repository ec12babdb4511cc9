"""Stage launches that go through the patches in alternating directions, with
states streamed out or left in the caches by their size."""
import numpy as np
import pytest

import amrhip

pytestmark = pytest.mark.gpu


def uniform(n, level, ninst, scheme):
    """ninst periodic boxes of 4**level patches, their vortices in different places"""
    forests = []
    for k in range(ninst):
        f = amrhip.Forest(1, 1, (1, 1), 0.0, 0.0, 1.0, n, level, level)
        f.apply_ic(amrhip.vortex_ic(0.1, 0.4 + 0.05 * k, 0.5))
        forests.append(f)
    insts = [amrhip.make_inst(1.0, (0,) * 4, 0.2, 1e-5) for _ in forests]
    arrays = amrhip.batch_external(forests)
    g = amrhip.Gpu()
    g.setup(n, scheme, insts, *arrays[:4], arrays[4])
    return g


# one size on each side of each line of the rule: 40 MB of vectors (two vectors of
# SSP-RK2, three of SSP-RK3 and LSERK45, four of RK4), 280 MB for the last two
@pytest.mark.parametrize("n,level,ninst,scheme,other", [
    (8, 6, 1, 3, (2, 4, 1)), (8, 6, 2, 3, (2, 4, 1)), (4, 8, 1, 2, (8, 1, 1)), (2, 9, 1, 1, (16, 1, 0)),
    (4, 8, 1, 5, (8, 1, 0)), (4, 8, 3, 5, (8, 1, 0)), (16, 5, 2, 5, (1, 4, 0)), (16, 6, 3, 5, (1, 4, 0)),
    (8, 7, 1, 4, (4, 4, 1)), (8, 7, 3, 4, (4, 4, 1))])
def test_large_states_equal_another_tile(n, level, ninst, scheme, other):
    """three steps of the default tile, whose odd and even launches run in
    opposite directions, against a tile that always streams: the same bits"""
    print(f"n={n} level={level} instances={ninst} scheme={scheme}", flush=True)
    g = uniform(n, level, ninst, scheme)
    q0 = g.soln()
    g.run(3)
    got = [g.soln(), *g.time()]
    g.set_tile(*other)
    g.upload(q0)
    g.set_time([0.0] * ninst)
    g.run(3)
    for a, b in zip(got, [g.soln(), *g.time()]):
        assert np.array_equal(a, b)
    g.close()


@pytest.mark.parametrize("n", [2, 4, 8, 16])
def test_norm_does_not_depend_on_the_direction(n):
    """the residual norm is summed in the patches' order whichever way a launch
    goes: one step of three stages from the same state twice"""
    g = uniform(n, 4, 1, 3)
    q0 = g.soln()
    for tile in amrhip.tile_variants(n):
        g.set_tile(*tile)
        norms = []
        for _ in range(2):
            g.upload(q0)
            g.set_time([0.0])
            norms.append(g.run(1))
        assert norms[0] == norms[1], tile
    g.close()


@pytest.mark.parametrize("graphs", [False, True])
@pytest.mark.parametrize("n,level", [(4, 3), (8, 3), (8, 8), (16, 2)])
def test_cfl_of_the_state_at_hand(n, level, graphs):
    """the CFL minimum turns through the sets of sub-slots: asked for several
    times in a row, between runs and after a new state, it is that of a context
    that holds this state alone, and the runs go on as they would without it"""
    g, ref = uniform(n, level, 2, 3), uniform(n, level, 2, 3)
    g.set_graphs(graphs)
    alone = uniform(n, level, 2, 3)
    for k in (1, 2, 3):
        g.run(k)
        ref.run(k)
        for _ in range(4):
            got = g.cfl()
        q = g.soln()
        assert np.array_equal(q, ref.soln())
        alone.upload(q)
        assert np.array_equal(got, alone.cfl())
    alone.upload(q * 1.25)
    g.upload(q * 1.25)
    assert np.array_equal(g.cfl(), alone.cfl())
    for c in (g, ref, alone):
        c.close()
