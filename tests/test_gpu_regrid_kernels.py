"""The kernels a regrid reads the resident state with (gradient indicator,
density tags, tagger features) at quadrant counts around their workgroups'
patches and with values at the edges of their arithmetic."""
import numpy as np
import pytest

import amrhip

pytestmark = pytest.mark.gpu


def forest(n, splits, seed):
    """a 2 x 1 brick, periodic in x, with `splits` quadrants of it refined in
    turn (3 more quadrants each, hanging faces), random positive states"""
    rng = np.random.default_rng(seed)
    f = amrhip.Forest(2, 1, (1, 0), 0.0, 0.0, 1.0, n, 0, 6)
    for k in range(splits):
        flags = np.zeros(f.nquad, np.int32)
        flags[(7 * k) % f.nquad] = 1
        f.refine(flags)
        f.balance()
    q = f.soln()
    q[..., 0] = np.exp(rng.uniform(-1.5, 1.0, q.shape[:3]))
    q[..., 1:3] = rng.uniform(-1.0, 1.0, q.shape[:3] + (2,))
    q[..., 3] = rng.uniform(2.0, 5.0, q.shape[:3])
    return f


def context(f):
    g = amrhip.Gpu()
    g.setup(f.n, 3, [amrhip.make_inst(1.0)], *f.external())
    return g


@pytest.mark.parametrize("n", [2, 4, 8, 16])
@pytest.mark.parametrize("splits", [0, 1, 5, 24])
def test_indicator_and_tags(n, splits):
    """bit for bit the host's indicator; the density tags of the patch minima
    and maxima"""
    f = forest(n, splits, 10 * n + splits)
    print(f"n={n} quads={f.nquad}", flush=True)
    g = context(f)
    assert np.array_equal(g.indicator(), f.indicator())
    rho = f.soln()[..., 0].reshape(f.nquad, -1)
    lo, hi = float(np.median(rho.min(axis=1))), float(np.median(rho.max(axis=1)))
    exp = (rho.min(axis=1) <= lo) | (rho.max(axis=1) >= hi)
    assert np.array_equal(g.feature_tags([1, 2], [lo, hi]), exp.astype(np.int32))
    g.close()


@pytest.mark.parametrize("case", ["rest", "negative zeros", "tiny", "huge", "mixed scales", "single spike"])
def test_features_at_the_edges_of_the_quotient(oracle, case):
    """momenta that vanish, signed zeros, and scales outside the range the
    product form of the quotient covers: bit for bit the oracle's quotients"""
    f = forest(8, 9, 5)
    q = f.soln()
    if case == "rest":
        q[..., 1:3] = 0.0
    elif case == "negative zeros":
        q[..., 1] = -0.0
        q[..., 2] = np.where(np.arange(8) % 3 == 0, -0.0, q[..., 2])
    elif case == "tiny":
        q[...] *= 2.0 ** -500
    elif case == "huge":
        q[...] *= 2.0 ** 600
    elif case == "mixed scales":
        q[::2] *= 2.0 ** 450
        q[1::3, ..., 2] *= 2.0 ** -900
    else:
        q[..., 1] = 0.0
        q[:, 3, 5, 1] = -2.5e-7
    ci, fi, _, soln = f.external()
    g = context(f)
    exp = oracle.tagger_features(8, ci, fi, soln)
    assert np.array_equal(g.tagger_features(), exp)
    g.close()


@pytest.mark.parametrize("batch", [64, 2176, 4096, 6208])
def test_training_step_follows_the_gradient(batch):
    """minibatches whose partial sums span one, two and three chunks, the last
    one of 6208 rows part empty: from zero moments Adam moves every parameter
    by lr against its gradient's sign (the step is lr g / (|g| + eps)), and the
    loss it reports is the gradient call's"""
    from test_tagger_oracle import random_problem
    P, X, y, cw = random_problem(90, n=batch)
    m, lr = amrhip.Mlp(0), 1e-3
    m.set_params(P)
    loss, g = m.grad(X, y, cw)
    ts = amrhip.Tagset()
    ts.append(X, y)
    losses = m.train(ts, epochs=1, batch=batch, lr=lr, cw=cw, seed=1)
    step = m.params() - P
    # the two sum in other orders: FP32 sums of `batch` terms differ by a few
    # parts in 1e6 of the largest, so a gradient over 1e-3 of its block's
    # largest keeps its sign; the step is exact to the rounding of P
    big = np.abs(g) > 1e-3 * np.abs(g).max()
    assert big.sum() > 500
    assert np.allclose(step[big], -lr * np.sign(g[big]), rtol=0, atol=1e-6 + 2.0 ** -23 * np.abs(P).max())
    assert abs(losses[0] - loss) <= 1e-5 * abs(loss)
    m.close()
    ts.close()


@pytest.mark.parametrize("splits", [0, 1, 2, 24])
def test_broken_densities_8x8(splits):
    """NaN, infinite and zero densities in some cells, a whole patch of NaN: the
    indicator ignores a pair without a quotient and the tags a cell without a
    value, as the host's do, in a wave's first and last patch alike"""
    f = forest(8, splits, 70 + splits)
    q = f.soln()
    rng = np.random.default_rng(splits)
    for bad in (np.nan, np.inf, 0.0):
        q[..., 0][rng.uniform(size=q.shape[:3]) < 0.02] = bad
    if f.nquad > 1:
        q[f.nquad - 1, ..., 0] = np.nan
    g = context(f)
    assert np.array_equal(g.indicator(), f.indicator(), equal_nan=True)
    rho = f.soln()[..., 0].reshape(f.nquad, -1)
    with np.errstate(invalid="ignore"):
        exp = (rho <= 0.5).any(axis=1) | (rho >= 1.4).any(axis=1)
    assert np.array_equal(g.feature_tags([1, 2], [0.5, 1.4]), exp.astype(np.int32))
    g.close()


@pytest.mark.parametrize("scale", [0, -450, 500])
def test_features_round_through_fp32(oracle, scale):
    """quotients just above and below the middle of two BF16 values, closer to it
    than FP32 tells: they are rounded to FP32 first and then, a tie, to even, in
    the range of the product form of the quotient and outside it"""
    f = forest(8, 3, 11)
    q = f.soln()
    k = np.arange(64).reshape(8, 8)
    mid = 0.5 + (2 * (k % 32) + 1) * 2.0 ** -9           # ties between neighbours in BF16
    for c, eps in ((1, 2.0 ** -31), (2, -2.0 ** -31), (3, 2.0 ** -28)):
        q[..., c] = (mid + eps) * 2.0 ** scale
        q[:, 0, 0, c] = 2.0 ** scale                     # the maximum
    ci, fi, _, soln = f.external()
    g = context(f)
    assert np.array_equal(g.tagger_features(), oracle.tagger_features(8, ci, fi, soln))
    g.close()
