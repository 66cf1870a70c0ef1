"""The cell-grouped push of the mixed-precision family (3D, and 2D at order 3) at the sizes where it can
go wrong, one PPC step against the FP64 oracle on inputs that FP32 holds exactly: boxes no segment
divides, rows that hold many cells, a crowded cell, segments of many work items, particles that leave the
tile in numbers beyond the list of the one-by-one push, segment shapes without the fixed stage. Moments
within 1e-5, the bound of the family's other one-step tests."""
import numpy as np
import pytest

import oracle_lib as O
import parity_util as U
from phare_amd import phx

pytestmark = pytest.mark.gpu

# name: cells, particles per cell, speed (cells per half step, standard deviation), tuning, orders
LAYOUTS = {
    "ragged": ((9, 11, 13), 8, 0.05, {}, (1, 2, 3)),
    "crowded": ((9, 10, 9), 8, 0.05, {}, (1, 2, 3)),
    "fast": ((12, 12, 12), 60, 0.9, {}, (1, 2, 3)),
    "shape": ((10, 9, 16), 12, 0.05, dict(segment_shape=[2, 4, 8]), (1, 2, 3)),
    "ragged2d": ((9, 35), 10, 0.05, {}, (3,)),
    "items2d": ((10, 37), 90, 0.05, dict(rows_per_item=3), (3,)),
    "fast2d": ((12, 40), 100, 0.9, {}, (3,)),
    "line2d": ((10, 65), 12, 0.05, dict(segment_shape=[1, 64]), (3,)),
}


@pytest.mark.parametrize("layout,order", [(k, o) for k, v in LAYOUTS.items() for o in v[4]])
def test_one_step(layout, order):
    print(f"[gpu] FP32 cell push {layout} order {order}", flush=True)
    ncells, ppc, speed, tuning, _ = LAYOUTS[layout]
    dim = len(ncells)
    rng = np.random.default_rng(100 * order + len(layout))
    dx = [0.3, 0.25, 0.2][:dim]
    n = ppc * int(np.prod(ncells))
    p = U.random_particles(rng, dim, n, ncells, [0] * dim, 0)
    if layout == "crowded":
        p["icell"][:1500] = (4, 5, 3)
    dt = 0.01
    # no move of two cells in a half step, and less than one cell per step where the particle
    # could leave the ghost layer
    inner = np.all((p["icell"] >= 4) & (p["icell"] < np.array(ncells) - 4), axis=1) & (speed > 0.5)
    most = np.where(inner, 0.9, 0.4)[:, None]
    p["v"] = np.clip(speed * rng.standard_normal((n, 3)), -most, most) * np.array([0.3, 0.25, 0.2]) / (0.5 * dt)
    p["charge"] = np.ones(n)
    for k in ("delta", "v", "weight"):
        p[k] = np.minimum(p[k], np.float32(1) - np.finfo(np.float32).epsneg) if k == "delta" else p[k]
        p[k] = p[k].astype(np.float32).astype(np.float64)
    g = phx.Level(dim, order, ncells, dx, capacity=n, precision=phx.PRECISION_FP32, apply_tuning_table=False)
    o = O.Sim(dim, order, ncells, dx)
    if tuning:
        g.set_tuning(**tuning)
    for k in range(3):
        b = np.full(g.shape(phx.F_B + k), 0.1 * (k + 1))
        g.set(phx.F_B + k, b)
        o.set(O.F_B + k, b)
    g.set_particles(0, phx.DOMAIN, p)
    o.set_particles(0, 0, p)
    g.initialize()
    o.initialize()
    g.advance(dt, 1)
    o.advance(dt, 1)
    for k in range(5):
        U.assert_close(g.get(phx.f_pop(0, k)), o.get(O.f_pop(0, k)), 1e-5, what=f"moment {k}")
    assert g.diagnostics()["count"] == o.diagnostics()["count"]
    g.close()
