"""The cell-grouped 3D push (k_push_cell: the particles of one cell deposit together on the matrix
cores, E/B gathered from a stage in LDS) at the sizes where it can go wrong, against the oracle at
1e-12: boxes no segment divides, rows that hold many cells, a crowded cell, segments shared by several
workgroups, particles that leave the tile or the domain in numbers beyond the list of the one-by-one
push, a segment shape without the fixed stage, one charge and mixed charges, and the drop-in updater on
sorted storage in both modes."""
import sys

import numpy as np
import pytest

import oracle_lib as O
import parity_util as U
from phare_amd import phx

pytestmark = pytest.mark.gpu

# name: cells, particles per cell, speed (cells per half step, standard deviation), segment shape
LAYOUTS = {
    "ragged": ((9, 11, 13), 3, 0.05, None),
    "crowded": ((9, 10, 9), 2, 0.05, None),
    "shared": ((12, 9, 12), 90, 0.05, None),
    "fast": ((12, 12, 12), 60, 0.9, None),
    "shape": ((10, 9, 16), 12, 0.1, [2, 4, 8]),
}


def _pair(layout, order, charges):
    ncells, ppc, speed, shape = LAYOUTS[layout]
    rng = np.random.default_rng(100 * order + len(layout))
    dx = [0.3, 0.25, 0.2]
    n = ppc * int(np.prod(ncells))
    p = U.random_particles(rng, 3, n, ncells, [0, 0, 0], 0)
    if layout == "crowded":
        p["icell"][:1500] = (4, 5, 3)
    dt = 0.05
    # no move of two cells in a half step, and less than one cell per step where the particle
    # could leave the ghost layer (the innermost segment alone scatters over its neighbours)
    inner = np.all((p["icell"] >= 4) & (p["icell"] < 8), axis=1) & (layout == "fast")
    most = np.where(inner, 0.95, 0.4)[:, None]
    step = np.clip(speed * rng.standard_normal((n, 3)), -most, most)
    p["v"] = step * np.array(dx) / (0.5 * dt)
    p["charge"] = np.ones(n) if charges == "one" else np.where(rng.random(n) < 0.5, 1.0, 2.0)
    g = phx.Level(3, order, ncells, dx, capacity=n, apply_tuning_table=False)
    o = O.Sim(3, order, ncells, dx)
    if shape:
        g.set_tuning(segment_shape=shape)
    for k in range(6):
        a = 0.02 * rng.standard_normal(g.shape(phx.F_EAVG + k)) + (0.3 if k == 4 else 0.0)
        g.set(phx.F_EAVG + k, a)
        o.set(O.F_EAVG + k, a)
    g.set_particles(0, phx.DOMAIN, p)
    o.set_particles(0, 0, p)
    g.sort_particles()
    return g, o, dt


@pytest.mark.parametrize("charges", ["one", "mixed"])
@pytest.mark.parametrize("order", [1, 2, 3])
@pytest.mark.parametrize("layout", list(LAYOUTS))
def test_move_ions_on_sorted_storage(layout, order, charges):
    print(f"[gpu] cell push {layout} order {order} charges {charges}", flush=True)
    sys.stdout.flush()
    g, o, dt = _pair(layout, order, charges)
    for mode in (phx.MODE_DOMAIN_ONLY, phx.MODE_ALL):
        g.move_ions(dt, mode)
        o.move_ions(dt, mode)
        for k in range(5):
            U.assert_close(g.get(phx.f_pop(0, k)), o.get(O.f_pop(0, k)), what=f"mode {mode} moment {k}")
    U.assert_same_particles(g.get_particles(), o.get_particles())
    g.close()


@pytest.mark.parametrize("order", [1, 2, 3])
def test_drop_in_updater_on_sorted_storage(order):
    print(f"[gpu] cell push, drop-in updater order {order}", flush=True)
    g, o, dt = _pair("fast", order, "one")
    for mode in (phx.MODE_DOMAIN_ONLY, phx.MODE_ALL):
        g.update_populations(dt, mode)
        o.update_populations(dt, mode)
        for k in range(5):
            U.assert_close(g.get(phx.f_pop(0, k)), o.get(O.f_pop(0, k)), what=f"mode {mode} moment {k}")
    for kind, okind in ((phx.DOMAIN, 0), (phx.PATCH_GHOST, 1)):
        U.assert_same_particles(g.get_particles(0, kind), o.get_particles(0, okind), what=f"kind {kind}")
    g.close()
