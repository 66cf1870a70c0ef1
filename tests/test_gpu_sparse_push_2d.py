"""The 2D cell-grouped push on both sides of the densities at which its particles deposit lane by lane
(order 1 up to 14 slots per cell, order 2 up to 6.5, order 3 up to 3.75) and where its small groups do (order 1),
against the oracle: FP64 at 1e-12 with one charge and mixed charges, before and after a second sort, and
mixed precision (order 3) at 1e-5, the bounds of the other tests of these families."""
import numpy as np
import pytest

import oracle_lib as O
import parity_util as U
from phare_amd import phx

pytestmark = pytest.mark.gpu

CELLS, DX, DT = (11, 45), [0.3, 0.25], 0.05


def _particles(rng, ppc, charges):
    n = ppc * int(np.prod(CELLS))
    p = U.random_particles(rng, 2, n, CELLS, [0, 0], 0)
    # as many per cell everywhere, but for a crowded cell
    cells = np.stack(np.meshgrid(*[np.arange(m) for m in CELLS], indexing="ij"), -1).reshape(-1, 2)
    p["icell"] = np.repeat(cells, ppc, 0).astype(np.int32)
    p["icell"][:n // 16] = (5, 17)
    p["v"] = np.clip(0.15 * rng.standard_normal((n, 3)), -0.4, 0.4) * np.array([0.3, 0.25, 0.2]) / (0.5 * DT)
    p["charge"] = np.ones(n) if charges == "one" else np.where(rng.random(n) < 0.5, 1.0, 2.0)
    return p


@pytest.mark.parametrize("charges", ["one", "mixed"])
@pytest.mark.parametrize("order,ppc", [(1, 1), (1, 13), (1, 15), (2, 1), (2, 6), (2, 7), (3, 1), (3, 3), (3, 4)])
def test_fp64(order, ppc, charges):
    print(f"[gpu] sparse push order {order} {ppc} per cell, charges {charges}", flush=True)
    rng = np.random.default_rng(10 * order + ppc)
    p = _particles(rng, ppc, charges)
    g = phx.Level(2, order, CELLS, DX, apply_tuning_table=False)
    o = O.Sim(2, order, CELLS, DX)
    for k in range(6):
        a = 0.02 * rng.standard_normal(g.shape(phx.F_EAVG + k)) + (0.3 if k == 4 else 0.0)
        g.set(phx.F_EAVG + k, a)
        o.set(O.F_EAVG + k, a)
    g.set_particles(0, phx.DOMAIN, p)
    o.set_particles(0, 0, p)
    for _ in range(2):
        g.sort_particles()
        for mode in (phx.MODE_DOMAIN_ONLY, phx.MODE_ALL):
            g.move_ions(DT, mode)
            o.move_ions(DT, mode)
            for k in range(5):
                U.assert_close(g.get(phx.f_pop(0, k)), o.get(O.f_pop(0, k)), what=f"mode {mode} moment {k}")
    U.assert_same_particles(g.get_particles(), o.get_particles())
    g.close()


@pytest.mark.parametrize("ppc", [1, 3, 4])
def test_mixed_precision(ppc):
    print(f"[gpu] sparse push, mixed precision, {ppc} per cell", flush=True)
    rng = np.random.default_rng(ppc)
    p = _particles(rng, ppc, "one")
    for k in ("delta", "v", "weight"):
        p[k] = np.minimum(p[k], np.float32(1) - np.finfo(np.float32).epsneg) if k == "delta" else p[k]
        p[k] = p[k].astype(np.float32).astype(np.float64)
    g = phx.Level(2, 3, CELLS, DX, capacity=len(p["weight"]), precision=phx.PRECISION_FP32, apply_tuning_table=False)
    o = O.Sim(2, 3, CELLS, DX)
    for k in range(3):
        b = np.full(g.shape(phx.F_BAVG + k), 0.1 * (k + 1))
        g.set(phx.F_BAVG + k, b)
        o.set(O.F_BAVG + k, b)
    g.set_particles(0, phx.DOMAIN, p)
    o.set_particles(0, 0, p)
    g.sort_particles()
    for mode in (phx.MODE_DOMAIN_ONLY, phx.MODE_ALL):
        g.move_ions(DT, mode)
        o.move_ions(DT, mode)
        for k in range(5):
            U.assert_close(g.get(phx.f_pop(0, k)), o.get(O.f_pop(0, k)), 1e-5, what=f"mode {mode} moment {k}")
    assert g.diagnostics()["count"] == o.diagnostics()["count"]
    g.close()
