"""The push with 16, 8 and 4 wavefronts per tile (the launcher picks by the
number of tiles: up to 256, up to 768, more) against the oracle: boxes just
inside and past each limit, cells from empty to fuller than a wavefront.

FP64: cell counts equal, fields and energies to 1e-10 (as the parity tests
over more steps); FP32: energies to 1e-4."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(4, 4, 8), (32, 16, 32), (34, 16, 32), (32, 48, 32), (34, 48, 31)])
def test_push_by_tiles(picmod, orc, n):
    rng = np.random.default_rng(n[0] + n[2])
    L = tuple(0.1 * k for k in n)
    cells = np.stack(np.meshgrid(*[np.arange(k) for k in n], indexing="ij")).reshape(3, -1)
    few = cells.shape[1] > 1000
    parts = []
    for sort, m, qm, drift in ((0, 0.02, 1 / 1836.0, 0.0), (1, -0.02, -1.0, 0.3)):
        per = rng.choice((0, 1, 2, 3) if few else (0, 1, 7, 90), cells.shape[1])
        at = np.repeat(cells, per, axis=1)
        x = (at + rng.uniform(1e-6, 1 - 1e-6, at.shape)) * 0.1
        p = rng.normal(0.0, 0.1, at.shape)
        p[0] += drift
        parts.append((sort, *x, *p, m, qm))
    o = orc.Oracle(n, L, 0.04)
    g64, g32 = [picmod.Pic(picmod.make_params(n, L, 0.04, precision=k, departure_cap=0))
                for k in (0, 1)]
    for q in (o, g64, g32):
        for a in parts:
            q.load_particles(*a)
    for nt in range(1, 6):
        o.step(nt)
        e64, e32 = g64.step(nt), g32.step(nt)
        e = o.energy()
        assert abs(e64 - e) <= 1e-10 * e
        assert abs(e32 - e) <= 1e-4 * e
        assert np.array_equal(g64.cell_counts(), np.asarray(o.cell_counts()).reshape(-1))
    for k in range(9):
        a, b = np.asarray(o.get_field(k)).reshape(-1), g64.get_field(k)
        assert np.abs(a - b).max() <= 1e-10 * max(np.abs(a).max(), 1e-300), k
    assert g32.particle_count() == g64.particle_count() == o.particle_count()
    g64.close()
    g32.close()
