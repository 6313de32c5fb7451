"""FP64 adjoint of a particle that lands exactly on the upper face of its cell.
Such a particle stays in the cell (the reference's flyDirection tests v > v0 +
h), and the next step reads the nodes behind the face: in a tile's last cell the
outermost plane of the tile's box.

The same cluster of particles once with that cell last in its tile and once one
cell lower, inside the tile: the two gradients differ by rounding only.  (The
energy counts the ghost nodes too, so the nodes that lie within the run's three
steps of the box's faces are left out.)  Every contribution to a current node is rounded to
2^-48 (up to 41 particles with two pieces each, fields of about 0.1), which
leaves about 1e-11 of the largest entry; 1e-9 is allowed."""
from fractions import Fraction

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

N, H, TAU = (16, 16, 24), 0.125, 0.0625
LAST = (7, 7, 15)        # last cell of a 2 x 4 x 8 tile along each axis


def start_of(face):
    """where a free particle of momentum 0.75 starts to land on the face: the
    end is fma(tau/gamma, p, x) with 1/gamma = 0.8"""
    move = Fraction(TAU * 0.8) * Fraction(0.75)
    x = float(Fraction(face) - move)
    for v in (x, np.nextafter(x, 0.0), np.nextafter(x, 1.0)):
        if float(Fraction(float(v)) + move) == face:
            return float(v)
    raise AssertionError("no start lands on the face")


def cluster(axis, shift):
    """(sort, m, q_m, positions, momenta) with the face particle first"""
    rng = np.random.default_rng(5 + axis)
    base = np.array(LAST, dtype=float)
    u = np.round(rng.uniform(-2.0, 2.0, (40, 3)) * 2.0**30) / 2.0**30
    x = (base + 0.5 + u) * H
    p = rng.normal(0.0, 0.3, (40, 3))
    x[:, axis] += shift * H
    face = (LAST[axis] + 1 + shift) * H
    x0 = (base + (0.3, 0.4, 0.6)) * H
    x0[axis] = start_of(face)
    p0 = np.zeros(3)
    p0[axis] = 0.75
    return face, [(1, -1.0, -1.0, x0[None], p0[None]), (2, -0.5, -1.0, x[:20], p[:20]),
                  (0, 1.0, 1.0 / 1836.0, x[20:], p[20:])]


@pytest.mark.parametrize("axis", [0, 1, 2])
def test_gradient_of_a_particle_on_its_cells_upper_face(picmod, axis):
    out = []
    for shift in (-1, 0):
        face, parts = cluster(axis, shift)

        def ctx():
            g = picmod.Pic(picmod.make_params(N, tuple(k * H for k in N), TAU, departure_cap=0,
                                              differentiable=1, ghost_mode=1))
            for sort, m, q_m, x, p in parts:
                g.load_particles(sort, *x.T.copy(), *p.T.copy(), m, q_m)
            return g

        g = ctx()
        g.run(1, 1)
        at = g.particles()
        k = int(np.flatnonzero(g.particle_ids() == 0)[0])
        assert at["xyz"[axis]][k] == face                     # on the face, and still in the cell
        cell = np.unravel_index(at["cell"][k], N)
        assert cell[axis] == LAST[axis] + shift
        g.close()
        g = ctx()
        g.forward_record(3, 3)
        rng = np.random.default_rng(9)
        seed = {q: rng.normal(size=g.id_count()) for q in ("x", "y", "z", "px", "py", "pz")}
        out.append(g.adjoint(weights=np.ones(3), seed=seed))
        g.close()
    for q in ("x", "y", "z", "px", "py", "pz"):
        a, b = (np.asarray(o[q]) for o in out)
        assert np.abs(a - b).max() <= 1e-9 * np.abs(a).max(), q
    for q in ("Ex", "Ey", "Ez", "Hx", "Hy", "Hz"):
        sh = tuple(k + 2 for k in N)
        a, b = (np.asarray(o[q]).reshape(sh) for o in out)
        inner = slice(5, N[axis] - 3)
        a = np.roll(a, 1, axis).swapaxes(0, axis)[inner]
        b = b.swapaxes(0, axis)[inner]
        assert np.abs(a - b).max() <= 1e-9 * np.abs(a).max(), q
