"""The FP64 differentiable form deposits the current in fixed point that holds a
contribution below 8: a step with a larger one is refused, a step with none is
not, also for a particle that moves over many cells in one step (its segment
then leaves the dual cell that it is deposited from, and the weights exceed the
cell's face)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

H, N = 0.1, (24, 24, 10)


def contributions(x, u, tau):
    """The 12 node contributions (cell.h:1511-1693) of a unit charge on the
    straight path x -> x + tau u, all of it from the dual cell of its start."""
    a = x / H - np.floor(x / H)
    b = a + tau * u / H
    d = 0.5 * (a + b) + 0.5 - np.floor(a + 0.5)
    D = b - a
    out = []
    for k in range(3):
        e, f = [q for q in range(3) if q != k]
        s = D[e] * D[f] / 12.0
        for i in (0, 1):
            for j in (0, 1):
                w = (d[e] if i else 1.0 - d[e]) * (d[f] if j else 1.0 - d[f])
                out.append(H * D[k] / tau * (w + s if i == j else w - s))
    return np.array(out)


# inside the dual cell; along x and y 5 cells, along all axes 2 to 4
@pytest.mark.parametrize("u,tau", [((0.5, 0.2, -0.1), 0.03), ((0.5, 0.5, 0.0), 1.0),
                                   ((-0.55, 0.5, 0.3), 0.75)])
@pytest.mark.parametrize("scale", [0.98, 1.02])
def test_refused_from_eight_on(picmod, u, tau, scale):
    u = np.array(u)
    x = (np.array([12, 12, 5]) + (0.1, 0.2, 0.3)) * H
    p = u / np.sqrt(1.0 - u @ u)
    m = scale * 8.0 / np.abs(contributions(x, u, tau)).max()
    g = picmod.Pic(picmod.make_params(N, tuple(k * H for k in N), tau, departure_cap=0,
                                      differentiable=1, ghost_mode=1))
    g.load_particles(1, *x[:, None], *p[:, None], m, -1.0)
    if scale < 1.0:
        g.run(1, 1)
    else:
        with pytest.raises(picmod.PicError) as e:
            g.run(1, 1)
        assert e.value.code == 8                      # PIC_ERR_CELL_RANGE
    g.close()
