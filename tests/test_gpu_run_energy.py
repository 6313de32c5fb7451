"""The energies of a run against single steps, bit for bit: a run leaves each
energy's partials to the next step's first launch and adds them up 32 steps at a
time, a single step sums its own.  Fewer steps than a batch, whole batches, one
more, a grid of exactly 1024 blocks of nodes (the last that defers) and one of
more; both forms whose current has no order; and a run that a step ends with an
error, whose energies up to that step are there."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _pair(picmod, n, precision, cap=0, drift=0.3, spread=0.1):
    L = tuple(0.1 * k for k in n)
    rng = np.random.default_rng(n[0])
    P = 20_000
    x = rng.uniform(1e-7, 1 - 1e-7, (3, P)) * np.array(L)[:, None]
    p = rng.normal(0.0, spread, (3, P))
    p[0] += drift
    out = []
    for _ in range(2):
        g = picmod.Pic(picmod.make_params(n, L, 0.04, precision=precision, departure_cap=cap,
                                          differentiable=1, ghost_mode=1))
        g.load_particles(0, *x, *np.zeros((3, P)), 1e-3, 1 / 1836.0)
        g.load_particles(1, *x, *p, -1e-3, -1.0)
        out.append(g)
    return out


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("n,steps", [((8, 8, 8), (1, 2, 31, 32, 33, 65)), ((62, 62, 62), (3,)),
                                     ((62, 62, 63), (3,))])
def test_run_equals_steps(picmod, n, steps, precision):
    a, b = _pair(picmod, n, precision)
    nt = 1
    for k in steps:
        wa = a.run(nt, k)
        wb = np.array([b.step(nt + s) for s in range(k)])
        nt += k
        assert np.array_equal(wa, wb), k
        for f in range(9):
            assert np.array_equal(a.get_field(f), b.get_field(f)), (k, f)
    wa, wb = a.forward_record(35, 20), b.run(nt, 35)
    assert np.array_equal(wa, wb)
    a.close()
    b.close()


@pytest.mark.parametrize("precision", [0, 1])
def test_energies_up_to_a_failing_step(picmod, precision):
    # particles gather speed until more leave a cell in a step than the cap allows
    a, b = _pair(picmod, (8, 8, 8), precision, cap=12, drift=0.0, spread=0.01)
    for g in (a, b):
        g.load_field(picmod.EX, np.full(g.G, 0.4))
    wa, wb = np.full(60, -1.0), np.full(60, -1.0)
    dp = C.POINTER(C.c_double)
    ra = a.lib.pic_run(a._ctx, 1, 60, wa.ctypes.data_as(dp))
    for s in range(60):
        rb = b.lib.pic_step(b._ctx, 1 + s, wb[s:].ctypes.data_as(dp))
        if rb:
            break
    assert ra == rb == 4                   # PIC_ERR_TOO_MANY_PARTICLES
    assert s > 0 and wb[s] != -1.0 and (wb[s + 1:] == -1.0).all()
    assert np.array_equal(wa, wb)
    a.close()
    b.close()
