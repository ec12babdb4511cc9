"""Steps with walls whose state depends on position and time (types 3-5), on the
tiles whose first stage forms the step's dt and so reads the step's start time
from another place than the stages after it."""
import ctypes

import numpy as np
import pytest

import amrhip
import pyoracle
from conftest import parity_err
from test_gpu_parity import RHS_TOL, TRAJ_TOL, dmr_forest, dmr_oracle_params

pytestmark = pytest.mark.gpu


def contexts(n, scheme, tiles, seed=5):
    arrays = dmr_forest(seed, n).external()
    gs = []
    for tile in tiles:
        g = amrhip.Gpu()
        g.setup(n, scheme, [amrhip.dmr_inst(1.0, 0.3, 2e-4 if scheme == 2 else 1.0)], *arrays)
        g.set_tile(*tile)
        gs.append(g)
    return arrays, gs


@pytest.mark.parametrize("t", [0.0, 0.07])
def test_rhs_of_2x2_patches(oracle, t):
    """every 2x2 tile against the oracle"""
    arrays, (g,) = contexts(2, 3, [(16, 3, 3)], 4)
    g.set_time([t])
    ref = oracle.rhs(dmr_oracle_params(oracle, t, 2), *arrays)
    for tile in amrhip.tile_variants(2):
        g.set_tile(*tile)
        assert parity_err(g.rhs(), ref) <= RHS_TOL
    g.close()


@pytest.mark.parametrize("scheme", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("n,own,other", [(2, (16, 3, 3), (16, 1, 0)), (4, (4, 3, 3), (8, 1, 1)), (4, (8, 3, 3), (8, 1, 0)),
                                          (8, (1, 5, 1), (2, 4, 1)), (16, (1, 5, 1), (1, 4, 0))])
def test_steps_equal_those_with_a_dt_kernel_ahead(n, own, other, scheme):
    """bit for bit, also where the time was set back since the last step"""
    _, gs = contexts(n, scheme, (own, other))
    for k, t in ((1, None), (3, 0.05), (1, 0.02), (2, None)):
        for g in gs:
            if t is not None:
                g.set_time([t])
            g.run(k)
        for a, b in zip([gs[0].soln(), *gs[0].time()], [gs[1].soln(), *gs[1].time()]):
            assert np.array_equal(a, b)
    for g in gs:
        g.close()


@pytest.mark.parametrize("n,tile", [(2, (16, 3, 3)), (4, (4, 3, 3)), (16, (1, 5, 1))])
def test_trajectory_against_oracle(oracle, n, tile):
    """10 SSP-RK3 steps from a time at which the shock stands on the top wall"""
    (ci, fi, geom, soln), (g,) = contexts(n, 3, [tile])
    t = 0.03
    g.set_time([t])
    g.run(10)
    q, work = np.array(soln, float), np.zeros(5 * soln.size)
    for _ in range(10):
        p = dmr_oracle_params(oracle, t, n)
        dt = oracle.time_step(p, ci, geom, q, 1.0)
        oracle.L.orc_rk_step(ctypes.byref(p), ci.size // 3, pyoracle.ipt(ci), pyoracle.dpt(geom), fi.size // 11,
                             pyoracle.ipt(fi), q.size, dt, pyoracle.dpt(q), pyoracle.dpt(work))
        t += dt
    assert g.time()[0][0] == pytest.approx(t, rel=1e-13)
    assert parity_err(g.soln(), q) <= TRAJ_TOL
    g.close()
