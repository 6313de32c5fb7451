"""The diagnostics kernels against the same sums in numpy, on boxes that no
tile divides and with bucket counts around the lanes of a group (0, 1, 15,
16, 17, 40 particles in a cell), both forms, before any step.

Tolerances: rho is a sum of n contributions each rounded to 2^-40 (error
2^-41), so n 2^-41, with n at most eight times the particles of the 27 cells
around a centre; the FP32 form's positions are rounded to 2^-24 of a cell,
which moves a weight by at most 3 x 2^-24.  The moments are FP64 sums of at
most a few thousand terms of order one: 1e-12 of the largest; FP32 momenta
add 2^-24 each, 1e-6."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

COUNTS = (0, 1, 15, 16, 17, 40)


def draw(n, rng):
    cells = np.stack(np.meshgrid(*[np.arange(k) for k in n], indexing="ij")).reshape(3, -1)
    out = []
    for sort, m, qm in ((0, 0.03, 1.0 / 1836.0), (1, -0.02, -1.0), (2, -0.001, -1.0)):
        per = rng.choice(COUNTS, cells.shape[1])
        at = np.repeat(cells, per, axis=1)
        x = (at + rng.uniform(1e-6, 1 - 1e-6, at.shape)) * 0.1
        p = rng.normal(0.0, 0.3, at.shape)
        out.append((sort, x, p, m, qm, at))
    return out


def rho_of(n, parts):
    r = np.zeros(n)
    for _, x, _, m, _, _ in parts:
        u = x / 0.1
        lo = np.floor(u - 0.5)
        far = u - 0.5 - lo
        for q in range(8):
            one = [(q >> d) & 1 for d in range(3)]
            w = m
            for d in range(3):
                w = w * (far[d] if one[d] else 1 - far[d])
            idx = tuple(((lo[d] + one[d]) % n[d]).astype(int) for d in range(3))
            np.add.at(r, idx, w)
    return r


@pytest.mark.parametrize("n", [(3, 3, 3), (5, 7, 9), (4, 9, 17)])
@pytest.mark.parametrize("precision", [0, 1])
def test_diagnostics_on_ragged_boxes(picmod, n, precision):
    rng = np.random.default_rng(sum(n) + precision)
    parts = draw(n, rng)
    params = picmod.make_params(n, tuple(0.1 * k for k in n), 0.04, precision=precision)
    with picmod.Pic(params) as g:
        for sort, x, p, m, qm, _ in parts:
            assert g.load_particles(sort, *x, *p, m, qm) == 0
        E = [rng.normal(0, 0.1, g.shape).astype(np.float32).astype(float) for _ in range(3)]
        for k in range(3):
            g.load_field(k, E[k])
        d0, res = g.gauss_residual(want_array=True)
        assert d0 == 0.0
        div = sum((e[1:-1, 1:-1, 1:-1] - np.roll(e, 1, d)[1:-1, 1:-1, 1:-1]) / 0.1
                  for d, e in enumerate(E))
        want = div - rho_of(n, parts)
        most = 27 * 3 * max(COUNTS) * 8
        tol = most * 2.0 ** -41 + 1e-12 * np.abs(div).max()
        if precision:
            tol += 0.03 * 27 * 3 * max(COUNTS) * 3 * 2.0 ** -24
        assert np.abs(res.reshape(n) - want).max() <= tol
        # the drift from the first call's residual
        E[1] = E[1] + 0.25 * rng.integers(0, 2, g.shape)
        g.load_field(1, E[1])
        d1, res1 = g.gauss_residual(want_array=True)
        assert d1 == np.abs(res1 - res).max() > 0
        rel = 1e-6 if precision else 1e-12
        mom = g.moments()
        for sort, x, p, m, qm, at in parts:
            gm = np.sqrt(1 + (p * p).sum(0))
            u, kin = p / gm, m / qm * (p * p).sum(0) / (gm + 1)
            want = np.array([x.shape[1], *x.sum(1), *p.sum(1), kin.sum(), np.abs(p).sum()])
            assert np.abs(mom[sort] - want).max() <= rel * np.abs(want).max()
            c = np.ravel_multi_index(tuple(at), n)
            num = np.bincount(c, minlength=g.ncell)
            for op, v in (("density", [np.full(len(c), m)]), ("kinetic_energy", [kin]),
                          ("velocity", u / np.maximum(num, 1)[c]), ("current", m * u)):
                got = g.cell_moments(sort, op).reshape(len(v), -1)
                for a, b in zip(got, v):
                    s = np.bincount(c, b, minlength=g.ncell)
                    assert np.abs(a - s).max() <= rel * max(np.abs(s).max(), np.abs(b).max())
