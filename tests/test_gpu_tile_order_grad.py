"""The reverse sweep on tiles that hold from nothing to many times the mean,
taken fullest first, against the same sweep with every tile equally full, which
takes them in their own order: particles of weight 0, at rest, make up what a
tile lacks and change neither the run nor the gradient of the others.

Only the order of the FP64 additions into shared nodes differs: 1e-12 of the
largest entry is allowed (about 1000 additions a node); in the FP32 form such a
difference may turn the rounding of a value to float, 1e-6."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

H, TILE = 0.1, np.array([2, 4, 8])


def skewed(rng, n, P, width):
    u = rng.uniform(0.0, 1.0, (3, P))
    u[1:] = np.mod(rng.normal(0.5, width, (2, P)), 1.0)
    return np.clip(u, 1e-7, 1 - 1e-7) * (np.array(n) * H)[:, None]


def filling(rng, n, x):
    """positions that bring every tile of the box to the fullest one's load"""
    t = [-(-k // s) for k, s in zip(n, TILE)]
    tile = np.ravel_multi_index(((x / H).astype(int) // TILE[:, None]), t)
    load = np.bincount(tile, minlength=np.prod(t))
    at = np.array(np.unravel_index(np.repeat(np.arange(len(load)), load.max() - load), t))
    lo = at * TILE[:, None]
    hi = np.minimum(lo + TILE[:, None], np.array(n)[:, None])
    return (lo + (hi - lo) * rng.uniform(0.01, 0.99, lo.shape)) * H, load


# tiles that the box fills and does not; 120 and 27 tiles
@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("n,width", [((8, 24, 40), 0.1), ((5, 10, 19), 0.15)])
def test_gradient_in_both_orders(picmod, n, width, precision):
    rng = np.random.default_rng(n[2])
    P = 20_000
    x = skewed(rng, n, P, width)
    p = rng.normal(0.0, 0.1, (3, P))
    p[0] += 0.3
    fill, load = filling(rng, n, x)
    assert load.max() > 2.5 * load.mean()
    out = []
    for even in (False, True):
        g = picmod.Pic(picmod.make_params(n, tuple(H * k for k in n), 0.04, precision=precision,
                                          departure_cap=0, differentiable=1, ghost_mode=1))
        g.load_particles(1, *x, *p, -1e-3, -1.0)
        if even:
            g.load_particles(0, *fill, *np.zeros_like(fill), 0.0, 1 / 1836.0)
        W = g.forward_record(6, 3)
        grad = g.adjoint(weights=np.ones(6))
        out.append((W, {k: np.array(v) for k, v in grad.items()}))
        g.close()
    (wa, ga), (wb, gb) = out
    assert np.array_equal(wa, wb)
    for k in ga:
        a, b = ga[k], gb[k][:len(ga[k])]
        assert np.abs(a - b).max() <= (1e-6 if precision else 1e-12) * np.abs(a).max(), k
