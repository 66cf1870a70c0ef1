"""Border sum and max over the periodic images, all moments in one launch, at the smallest periodic box
(2 g + 1 cells: every node has an image) and one cell more, two populations: bit for bit the oracle's."""
import numpy as np
import pytest

import oracle_lib as O
import parity_util as U
from phare_amd import phx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("extra", [1, 2])
@pytest.mark.parametrize("dim,order", [(1, 1), (1, 3), (2, 1), (2, 2), (3, 1), (3, 2)])
def test_border_fills_of_the_smallest_boxes(dim, order, extra):
    print(f"[gpu] border fills dim={dim} order={order} extra={extra}", flush=True)
    rng = np.random.default_rng(50 + 10 * dim + order)
    n = [2 * {1: 2, 2: 4, 3: 4}[order] + extra + (d == 1) for d in range(dim)]
    dx = [0.3, 0.25, 0.2][:dim]
    g = phx.Level(dim, order, n, dx, masses=(1.0, 4.0))
    o = O.Sim(dim, order, n, dx, masses=(1.0, 4.0))
    for p in (0, 1):
        for k in range(5):
            a = 0.5 + rng.random(g.shape(phx.f_pop(p, k)))
            g.set(phx.f_pop(p, k), a)
            o.set(O.f_pop(p, k), a)
    for s in (g, o):
        s.fill_moment_borders()
        s.update_ions()
        s.fill_ion_borders()
    for p in (0, 1):
        for k in range(5):
            U.assert_close(g.get(phx.f_pop(p, k)), o.get(O.f_pop(p, k)), rtol=0, what=f"pop {p} moment {k}")
    for fid in (25, 26, 27, 28, 29):
        U.assert_close(g.get(fid), o.get(fid), rtol=0, what=f"total {fid}")
    g.close()
