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
