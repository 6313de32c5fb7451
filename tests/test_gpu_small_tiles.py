"""The FP64 push on the 16-cell tiles of small boxes, and on either side of the
rule that picks them (by the tiles a CU gets), against the oracle: boxes down to
3x3x3, sides that no tile divides, cells from empty to fuller than a wavefront,
and a group that leaves its cell together.

Cell counts equal, fields and energies to 1e-10, as the parity tests over more
steps."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(3, 3, 3), (5, 7, 9), (32, 8, 8), (33, 9, 7), (64, 13, 11),
                               (64, 16, 16), (33, 24, 20), (36, 26, 33)])
def test_small_tiles(picmod, orc, n):
    rng = np.random.default_rng(sum(n))
    L = tuple(0.1 * k for k in n)
    cells = np.stack(np.meshgrid(*[np.arange(k) for k in n], indexing="ij")).reshape(3, -1)
    few = cells.shape[1] > 1000
    parts = []
    for sort, m, qm, drift in ((0, 0.02, 1 / 1836.0, 0.0), (1, -0.02, -1.0, 0.3)):
        per = rng.choice((0, 1, 2, 30) if few else (0, 1, 7, 90), cells.shape[1])
        at = np.repeat(cells, per, axis=1)
        x = (at + rng.uniform(1e-6, 1 - 1e-6, at.shape)) * 0.1
        p = rng.normal(0.0, 0.1, at.shape)
        p[0] += drift
        parts.append((sort, *x, *p, m, qm))
    # particles next to a cell's upper corner, all leaving together (the oracle
    # keeps the reference's storage of 48 departures a cell)
    x = np.array([[1.99], [1.98], [1.97]]) * 0.1 - rng.uniform(0, 1e-4, (3, 20))
    p = np.full((3, 20), 5.0)
    parts.append((2, *x, *p, -0.001, -1.0))
    o = orc.Oracle(n, L, 0.04)
    g = picmod.Pic(picmod.make_params(n, L, 0.04, departure_cap=0))
    for q in (o, g):
        for a in parts:
            q.load_particles(*a)
    for nt in range(1, 6):
        o.step(nt)
        e64, e = g.step(nt), o.energy()
        assert abs(e64 - e) <= 1e-10 * e
        assert np.array_equal(g.cell_counts(), np.asarray(o.cell_counts()).reshape(-1))
    for k in range(9):
        a, b = np.asarray(o.get_field(k)).reshape(-1), g.get_field(k)
        assert np.abs(a - b).max() <= 1e-10 * max(np.abs(a).max(), 1e-300), k
    assert g.particle_count() == o.particle_count()
    g.close()
