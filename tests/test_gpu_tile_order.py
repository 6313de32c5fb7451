"""The order in which the differentiable form takes its tiles (fullest first,
from the first checkpoint on) changes no result: a recorded run against a plain
run of the same particles, bit for bit, on boxes whose tiles hold from nothing
to many times the mean, with fewer and more tiles than the ordering's threads,
and on a uniform one.  The reverse sweep's recompute checks itself against the
checkpoints and must accept it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("n,width", [((4, 6, 9), 0.0), ((16, 36, 70), 0.08), ((6, 90, 41), 0.06),
                                     ((18, 33, 66), 0.0)])
def test_recorded_run_equals_plain_run(picmod, n, width, precision):
    rng = np.random.default_rng(n[1])
    L = np.array([0.1 * k for k in n])
    P = 120_000
    u = rng.uniform(0.0, 1.0, (3, P))
    if width:
        u[1:] = np.mod(rng.normal(0.5, width, (2, P)), 1.0)
    x = np.clip(u, 1e-7, 1 - 1e-7) * L[:, None]
    p = rng.normal(0.0, 0.1, (3, P))
    p[0] += 0.3
    out = []
    for recorded in (True, False):
        g = picmod.Pic(picmod.make_params(n, tuple(L), 0.04, precision=precision, departure_cap=0,
                                          differentiable=1, ghost_mode=1))
        g.load_particles(0, *x, *np.zeros((3, P)), 1e-3, 1 / 1836.0)
        g.load_particles(1, *x, *p, -1e-3, -1.0)
        W = g.forward_record(6, 3) if recorded else g.run(1, 6)
        out.append((W, [g.get_field(k) for k in range(9)], g.cell_counts()))
        if recorded:
            grad = g.adjoint(weights=np.ones(6))
            assert all(np.isfinite(np.asarray(v)).all() for v in grad.values())
        g.close()
    (wa, fa, ca), (wb, fb, cb) = out
    assert np.array_equal(wa, wb)
    assert np.array_equal(ca, cb)
    for a, b in zip(fa, fb):
        assert np.array_equal(a, b)
