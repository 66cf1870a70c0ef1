"""The drop-in updater after its first call in mode all, whose compaction leaves the segments of the last
sort behind each other without padding: the cell-grouped push over such arrays against the oracle at
1e-12, over three steps that add re-entering particles behind the segments and level ghosts that enter,
with one charge and mixed charges, a segment shape that leaves many segments empty, then after a sort
and after an upload of another array."""
import numpy as np
import pytest

import oracle_lib as O
import parity_util as U
from phare_amd import phx

pytestmark = pytest.mark.gpu

# cells, particles per cell, speed (cells per half step, standard deviation), tuning
LAYOUTS = {
    "2d": ((12, 37), 30, 0.12, {}),
    "2d-few": ((11, 40), 1, 0.12, dict(rows_per_item=1)),
    "2d-shape": ((13, 18), 12, 0.12, dict(segment_shape=[4, 16])),
    "3d": ((9, 11, 13), 6, 0.12, {}),
    "3d-empty": ((12, 10, 10), 1, 0.12, dict(segment_shape=[1, 1, 2])),
}


def _compare(g, o, mode):
    g.update_populations(0.05, mode)
    o.update_populations(0.05, mode)
    for k in range(5):
        U.assert_close(g.get(phx.f_pop(0, k)), o.get(O.f_pop(0, k)), what=f"mode {mode} moment {k}")
    for kind, okind in ((phx.DOMAIN, 0), (phx.PATCH_GHOST, 1), (phx.LEVEL_GHOST, 2)):
        U.assert_same_particles(g.get_particles(0, kind), o.get_particles(0, okind), what=f"kind {kind}")


@pytest.mark.parametrize("charges", ["one", "mixed"])
@pytest.mark.parametrize("order", [1, 2, 3])
@pytest.mark.parametrize("layout", list(LAYOUTS))
def test_updater_on_packed_segments(layout, order, charges):
    print(f"[gpu] packed push {layout} order {order} charges {charges}", flush=True)
    ncells, ppc, speed, tuning = LAYOUTS[layout]
    dim = len(ncells)
    rng = np.random.default_rng(100 * order + len(layout))
    dx = [0.3, 0.25, 0.2][:dim]

    def particles(n):
        p = U.random_particles(rng, dim, n, ncells, [0] * dim, 0)
        p["v"] = np.clip(speed * rng.standard_normal((n, 3)), -0.4, 0.4) * np.array([0.3, 0.25, 0.2]) / 0.025
        p["charge"] = np.ones(n) if charges == "one" else np.where(rng.random(n) < 0.5, 1.0, 2.0)
        return p

    n = ppc * int(np.prod(ncells))
    g = phx.Level(dim, order, ncells, dx, capacity=n, apply_tuning_table=False)
    o = O.Sim(dim, order, ncells, dx)
    if tuning:
        g.set_tuning(**tuning)
    for k in range(6):
        a = 0.02 * rng.standard_normal(g.shape(phx.F_EAVG + k)) + (0.3 if k == 4 else 0.0)
        g.set(phx.F_EAVG + k, a)
        o.set(O.F_EAVG + k, a)
    p = particles(n)
    lg = particles(200)
    lg["icell"][:, 0] = np.where(rng.random(200) < 0.5, -1, ncells[0])
    g.set_particles(0, phx.DOMAIN, p)
    o.set_particles(0, 0, p)
    g.sort_particles()
    for step in range(3):
        g.set_particles(0, phx.LEVEL_GHOST, lg)
        o.set_particles(0, 2, lg)
        _compare(g, o, phx.MODE_DOMAIN_ONLY)
        _compare(g, o, phx.MODE_ALL)
        # the leavers re-enter through the periodic image, behind the segments
        g.fill_ion_ghost_particles()
        dom, out = o.get_particles(0, 0), o.get_particles(0, 1)
        out["icell"] = out["icell"] % np.array(ncells)
        o.set_particles(0, 0, {k: np.concatenate([dom[k], out[k]]) for k in dom})
        o.set_particles(0, 1, {k: v[:0] for k, v in out.items()})
    g.sort_particles()
    _compare(g, o, phx.MODE_ALL)
    q = particles(n // 3)
    g.set_particles(0, phx.DOMAIN, q)
    o.set_particles(0, 0, q)
    _compare(g, o, phx.MODE_ALL)
    g.close()
