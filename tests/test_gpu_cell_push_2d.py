"""The cell-grouped push in 2D (k_push_cell<2>: one workgroup per work item of a segment) and the
split of segments into work items, at the sizes where they can go wrong, against the oracle at 1e-12:
boxes no segment divides, rows that hold many cells, a crowded cell, segments of many work items,
particles that leave the tile or the domain in numbers beyond the list of the one-by-one push, segment
shapes without the fixed stage, one charge and mixed charges, two populations whose arrays are cut
differently, and the drop-in updater on sorted storage in both modes."""
import numpy as np
import pytest

import oracle_lib as O
import parity_util as U
from phare_amd import phx

pytestmark = pytest.mark.gpu

# name: cells, particles per cell, speed (cells per half step, standard deviation), tuning
LAYOUTS = {
    "ragged": ((9, 11), 3, 0.05, {}),
    "crowded": ((9, 35), 2, 0.05, {}),
    "items": ((10, 37), 90, 0.05, dict(rows_per_item=3)),
    "fast": ((12, 40), 100, 0.9, {}),
    "shape": ((13, 18), 12, 0.05, dict(segment_shape=[4, 16])),
    "line": ((10, 65), 12, 0.05, dict(segment_shape=[1, 64])),
}


def _particles(layout, order, charges, pop):
    ncells, ppc, speed, _ = LAYOUTS[layout]
    rng = np.random.default_rng(100 * order + 10 * pop + len(layout))
    ppc = ppc if pop == 0 else 2
    n = ppc * int(np.prod(ncells))
    p = U.random_particles(rng, 2, n, ncells, [0, 0], 0)
    if layout == "crowded":
        p["icell"][:n // 2] = (4, 5)
    # no move of two cells in a half step, and less than one cell per step where the particle
    # could leave the ghost layer (the inner cells alone scatter over their neighbours)
    inner = np.all((p["icell"] >= 4) & (p["icell"] < np.array(ncells) - 4), axis=1) & (layout == "fast")
    most = np.where(inner, 0.95, 0.4)[:, None]
    step = np.clip(speed * rng.standard_normal((n, 3)), -most, most)
    p["v"] = step * np.array([0.3, 0.25, 0.2]) / (0.5 * 0.05)
    p["charge"] = np.ones(n) if charges == "one" else np.where(rng.random(n) < 0.5, 1.0, 2.0)
    return p


def _pair(layout, order, charges):
    ncells, _, _, tuning = LAYOUTS[layout]
    rng = np.random.default_rng(order)
    parts = [_particles(layout, order, charges, pop) for pop in range(2)]
    g = phx.Level(2, order, ncells, [0.3, 0.25], masses=[1.0, 2.0],
                  capacity=len(parts[0]["icell"]), apply_tuning_table=False)
    o = O.Sim(2, order, ncells, [0.3, 0.25], masses=[1.0, 2.0])
    if tuning:
        g.set_tuning(**tuning)
    for k in range(6):
        a = 0.02 * rng.standard_normal(g.shape(phx.F_EAVG + k)) + (0.3 if k == 4 else 0.0)
        g.set(phx.F_EAVG + k, a)
        o.set(O.F_EAVG + k, a)
    for pop, p in enumerate(parts):
        g.set_particles(pop, phx.DOMAIN, p)
        o.set_particles(pop, 0, p)
    g.sort_particles()
    return g, o


def _same(g, o, mode, call):
    getattr(g, call)(0.05, mode)
    getattr(o, call)(0.05, mode)
    for pop in range(2):
        for k in range(5):
            U.assert_close(g.get(phx.f_pop(pop, k)), o.get(O.f_pop(pop, k)),
                           what=f"mode {mode} population {pop} moment {k}")


@pytest.mark.parametrize("charges", ["one", "mixed"])
@pytest.mark.parametrize("order", [1, 2, 3])
@pytest.mark.parametrize("layout", list(LAYOUTS))
def test_move_ions_on_sorted_storage(layout, order, charges):
    print(f"[gpu] 2D cell push {layout} order {order} charges {charges}", flush=True)
    g, o = _pair(layout, order, charges)
    for mode in (phx.MODE_DOMAIN_ONLY, phx.MODE_ALL):
        _same(g, o, mode, "move_ions")
    g.sort_particles()
    for mode in (phx.MODE_DOMAIN_ONLY, phx.MODE_ALL):
        _same(g, o, mode, "move_ions")
    for pop in range(2):
        U.assert_same_particles(g.get_particles(pop), o.get_particles(pop))
    g.close()


@pytest.mark.parametrize("order", [1, 2, 3])
def test_drop_in_updater_on_sorted_storage(order):
    print(f"[gpu] 2D cell push, drop-in updater order {order}", flush=True)
    g, o = _pair("fast", order, "one")
    for mode in (phx.MODE_DOMAIN_ONLY, phx.MODE_ALL):
        _same(g, o, mode, "update_populations")
    for pop in range(2):
        for kind, okind in ((phx.DOMAIN, 0), (phx.PATCH_GHOST, 1)):
            U.assert_same_particles(g.get_particles(pop, kind), o.get_particles(pop, okind), what=f"kind {kind}")
    g.close()
