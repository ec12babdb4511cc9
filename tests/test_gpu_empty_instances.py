"""Instances without quadrants, whose dt and time no quadrant's wave keeps, beside
others that advance, leave and come back."""
import numpy as np
import pytest

import amrhip
from test_gpu_rows import small_forest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scheme", [1, 2, 3, 5])
@pytest.mark.parametrize("ninst", [3, 64, 65, 128, 129])
@pytest.mark.parametrize("n,own,other", [(4, (4, 3, 3), (8, 1, 1)), (8, (1, 5, 1), (2, 4, 1)), (16, (1, 5, 1), (1, 4, 0))])
def test_leave_and_come_back(n, own, other, ninst, scheme):
    """the first, a middle and the last instance leave, at first one of them,
    then all, then they come back: states, times and step sizes are bit for bit
    those of a tile that has a kernel for every instance's dt ahead of the step"""
    forest = small_forest(n, 7, True, 1, 2)
    live = sorted({0, ninst // 2, ninst - 1})
    insts = [amrhip.make_inst(1.0, (0,) * 4, 0.2, 1e-3 * (1 + k % 5), 2.5e-3 if k % 4 == 3 else 0.0)
             for k in range(ninst)]
    ci, fi, geom, soln, inst = amrhip.batch_external([forest] * len(live))
    inst = np.asarray(live, np.int32)[np.asarray(inst)]
    nq = forest.nquad

    def mesh_of(k):
        """the mesh of the first k of the live instances"""
        a = amrhip.batch_external([forest] * k)
        return a[0], a[1], inst[:k * nq]

    gs = []
    for tile in (own, other):
        g = amrhip.Gpu()
        g.setup(n, scheme, insts, ci, fi, geom, soln, inst)
        g.set_tile(*tile)
        gs.append(g)

    def run(k):
        for g in gs:
            g.run(k)
        for a, b in zip([gs[0].soln(), *gs[0].time()], [gs[1].soln(), *gs[1].time()]):
            assert np.array_equal(a, b)

    def remesh(to, src):
        c, f, i = mesh_of(to)
        for g in gs:
            g.remesh(c, f, np.asarray(src, np.int32), i)
        assert np.array_equal(gs[0].time()[1], gs[1].time()[1])

    run(2)
    remesh(2, np.arange(2 * nq))
    run(1)
    run(3)
    remesh(1, np.arange(nq))
    run(4)
    remesh(3, np.tile(np.arange(nq), 3))
    run(1)
    run(4)
    for g in gs:
        g.close()


@pytest.mark.parametrize("scheme", [2, 3])
@pytest.mark.parametrize("ninst", [3, 129])
@pytest.mark.parametrize("n,tile", [(4, (4, 3, 3)), (4, (8, 1, 1)), (8, (1, 5, 1)), (8, (2, 4, 1)), (16, (1, 5, 1)), (16, (1, 4, 0))])
def test_time_of_an_absent_instance_stays(n, tile, ninst, scheme):
    """an instance without quadrants does not advance: no last dt, and its time
    where it was, from a remesh or from the setup on, until it comes back"""
    forest = small_forest(n, 7, True, 1, 2)
    nq = forest.nquad
    live = [0, ninst - 1]
    insts = [amrhip.make_inst(1.0, (0,) * 4, 0.2, 1e-3) for _ in range(ninst)]
    ci, fi, geom, soln, inst = amrhip.batch_external([forest] * 2)
    inst = np.asarray(live, np.int32)[np.asarray(inst)]
    g = amrhip.Gpu()
    g.setup(n, scheme, insts, ci, fi, geom, soln, inst)
    g.set_tile(*tile)
    t0 = 0.25 * np.arange(ninst)
    g.set_time(t0)
    g.run(2)
    t, dt = g.time()
    absent = np.ones(ninst, bool)
    absent[live] = False
    assert np.array_equal(t[absent], t0[absent]) and not dt[absent].any()
    assert (t[live] > t0[live]).all() and (dt[live] > 0.0).all()
    one = amrhip.batch_external([forest])
    g.remesh(one[0], one[1], np.arange(nq, dtype=np.int32), np.zeros(nq, np.int32))
    assert g.time()[1][-1] == 0.0
    g.run(3)
    t1, dt1 = g.time()
    assert np.array_equal(t1[1:], t[1:]) and not dt1[1:].any() and t1[0] > t[0]
    g.remesh(ci, fi, np.tile(np.arange(nq, dtype=np.int32), 2), inst)
    g.run(1)
    t2, dt2 = g.time()
    assert np.array_equal(t2[absent], t0[absent]) and not dt2[absent].any()
    assert t2[-1] == t[-1] + dt2[-1] and dt2[-1] > 0.0
    g.close()
