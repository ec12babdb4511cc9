"""The row-marching stage kernel where its waves are least regular:
several patches share a wave, so instances, levels, stopped instances, walls
and the tail past the last patch meet inside one."""
import numpy as np
import pytest

import amrhip

pytestmark = pytest.mark.gpu


def small_forest(n, seed, periodic, lmin, lmax):
    rng = np.random.default_rng(seed)
    f = amrhip.Forest(1, 1, (int(periodic),) * 2, 0.0, 0.0, 1.0, n, lmin, lmax)
    for _ in range(lmax - lmin):
        f.refine((rng.uniform(size=f.nquad) < 0.3).astype(np.int32))
        f.balance()
    q = f.soln()
    rho, p = rng.uniform(0.5, 1.5, q.shape[:3]), rng.uniform(0.5, 1.5, q.shape[:3])
    u, v = rng.uniform(-0.3, 0.3, q.shape[:3]), rng.uniform(-0.3, 0.3, q.shape[:3])
    q[..., 0], q[..., 1], q[..., 2] = rho, rho * u, rho * v
    q[..., 3] = p / 0.4 + 0.5 * rho * (u * u + v * v)
    return f


@pytest.mark.parametrize("scheme", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("n", [2, 4])
def test_mixed_waves_equal_the_other_designs(n, scheme):
    """forests of 1, 4, and some tens to hundreds of quadrants batched so that
    waves hold patches of several instances, one instance stops after the
    first step, and the last wave is part empty: residual, states, times and
    step sizes are bit for bit those of every other tile"""
    forests = [small_forest(n, 1, True, 0, 0), small_forest(n, 2, False, 1, 1), small_forest(n, 3, False, 2, 4),
               small_forest(n, 4, True, 0, 0), small_forest(n, 5, False, 1, 4), small_forest(n, 6, True, 2, 3)]
    bcs = [(0, 0, 0, 0), (1, 2, 0, 1), (2, 1, 1, 0), (0, 0, 0, 0), (0, 1, 2, 1), (0, 0, 0, 0)]
    cap = 1e-3
    insts = [amrhip.make_inst(1.0, bc, 0.2, cap * (1 + k), 1e-9 if k == 2 else 0.0) for k, bc in enumerate(bcs)]
    arrays = amrhip.batch_external(forests)
    assert (arrays[0].size // 3) % (32 // n) != 0
    ref = None
    for tile in amrhip.tile_variants(n):
        print(f"n={n} scheme={scheme} tile={tile}", flush=True)
        g = amrhip.Gpu()
        g.setup(n, scheme, insts, *arrays[:4], arrays[4])
        g.set_tile(*tile)
        got = [g.rhs()]
        norm = g.run(3)
        got += [g.soln(), *g.time()]
        g.close()
        ref = ref or (tile, got, norm)
        for a, b in zip(got, ref[1]):
            assert np.array_equal(a, b), (tile, ref[0])
        # the norm sums each tile's workgroups in its own order
        assert abs(norm - ref[2]) <= 1e-12 * ref[2]


def test_default_tile_follows_the_mesh_until_one_is_set():
    """4x4 patches: the default takes four rows a step on a small mesh and two
    on a large one, also across a setup of another size; a tile that was set
    stays"""
    g = amrhip.Gpu()
    inst = [amrhip.make_inst(1.0, (0, 0, 0, 0), 0.2, 1e-3)]

    def setup(level):
        f = amrhip.Forest(1, 1, (1, 1), 0.0, 0.0, 1.0, 4, level, level)
        f.apply_ic(amrhip.vortex_ic(0.1, 0.5, 0.5))
        g.setup(4, 3, inst, *f.external())

    setup(3)
    assert g.tile() == (4, 3, 3)
    setup(8)
    assert g.tile() == (8, 3, 3)
    setup(2)
    assert g.tile() == (4, 3, 3)
    g.set_tile(8, 1, 0)
    setup(8)
    assert g.tile() == (8, 1, 0)
    g.close()


@pytest.mark.parametrize("scheme", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("n,own,other", [(2, (16, 3, 3), (16, 1, 0)), (4, (4, 3, 3), (8, 1, 1)), (4, (8, 3, 3), (8, 1, 0)),
                                          (8, (1, 5, 1), (2, 4, 1)), (16, (1, 5, 1), (1, 4, 0))])
def test_steps_without_a_prep_launch(n, own, other, scheme):
    """small meshes: the first stage forms the step's dt, in rotating sets of
    CFL sub-slots and two clocks; a tile that has a kernel ahead for it gives
    the same states, times and step sizes through runs of one and several
    steps, a CFL query, a new time, a new state, a remesh, an instance without
    quadrants, and a change to graph replay and back"""
    forests = [small_forest(n, 31, False, 1, 3), small_forest(n, 32, True, 1, 2), small_forest(n, 33, True, 0, 0)]
    insts = [amrhip.make_inst(1.0, (1, 0, 2, 1), 0.2, 2e-3), amrhip.make_inst(1.0, (0,) * 4, 0.15, 1e-3, 2.5e-3),
             # (SSP-RK2 takes the cap itself, not the CFL minimum: a stable one there)
             amrhip.make_inst(1.0, (0,) * 4, 0.25, 1.0 if scheme != 2 else 3e-3)]
    arrays = amrhip.batch_external(forests)
    nq = [f.nquad for f in forests]
    gs = []
    for tile in (own, other):
        g = amrhip.Gpu()
        g.setup(n, scheme, insts, *arrays[:4], arrays[4])
        g.set_tile(*tile)
        gs.append(g)

    def both(what):
        got = [what(g) for g in gs]
        a, b = ([np.asarray(x) for x in (r if isinstance(r, tuple) else (r,))] for r in got)
        for x, y in zip(a, b):
            assert np.array_equal(x, y)

    def state(g):
        return (g.soln(), *g.time())

    def run(k):
        for g in gs:
            g.run(k)
        both(state)

    run(1)
    run(4)
    both(lambda g: g.cfl())
    run(2)
    for g in gs:
        g.set_time([1e-4, 1e-3, 0.0])
    run(3)
    new = gs[0].soln() * 1.01
    for g in gs:
        g.upload(new)
    run(1)
    gs[0].set_graphs(True)
    run(3)
    gs[0].set_graphs(False)
    run(2)
    # the same mesh again, then without the last instance's quadrant
    ci, fi, _, _, inst = arrays
    src = np.arange(sum(nq), dtype=np.int32)
    for g in gs:
        g.remesh(ci, fi, src, inst)
    run(2)
    ci2, fi2, _, _, inst2 = amrhip.batch_external(forests[:2])
    for g in gs:
        g.remesh(ci2, fi2, src[:nq[0] + nq[1]], inst2)
    run(3)
    for g in gs:
        g.close()
