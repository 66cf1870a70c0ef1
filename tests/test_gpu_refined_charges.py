"""A finer level whose arrays hold refined particles of other charges than its uploads: the push and the
deposit over sorted and packed storage take every particle's own charge, against the oracle at 1e-12.
The coarser particles carry one other charge or mixed ones, and reach the finer domain array before the
sort, the level ghosts after it (those that enter join the domain array), or the level ghosts of a level
that has no upload yet; refined particles of the uploads' own charge are the case that changes nothing."""
import numpy as np
import pytest

import oracle_lib as O
import parity_util as U
from phare_amd import phx

pytestmark = pytest.mark.gpu

CELLS = {1: (30,), 2: (16, 14), 3: (13, 12, 11)}
DT = 0.05


def _particles(rng, dim, n, cells, lower, dx, charge):
    p = U.random_particles(rng, dim, n, cells, lower, 0)
    p["v"] = np.clip(0.1 * rng.standard_normal((n, 3)), -0.4, 0.4) * min(dx) / (0.5 * DT)
    p["charge"] = np.where(rng.random(n) < 0.5, 1.0, 2.0) if charge == "mixed" else np.full(n, charge)
    return p


@pytest.mark.parametrize("source", [1.0, 2.0, "mixed"])
@pytest.mark.parametrize("into", ["domain", "ghosts", "ghosts-first"])
@pytest.mark.parametrize("dim", [1, 2, 3])
def test_refined_particles_keep_their_charge(dim, into, source):
    print(f"[gpu] refined charges dim={dim} {into} source {source}", flush=True)
    order = 2
    rng = np.random.default_rng(dim)
    nc, dx = CELLS[dim], [0.4, 0.3, 0.3][:dim]
    h = [a / 2 for a in dx]
    flo, fhi = [6] * dim, [2 * n - 7 for n in nc]
    fn = [b - a + 1 for a, b in zip(flo, fhi)]
    coarse = phx.Level(dim, order, nc, dx, apply_tuning_table=False)
    coarse.set_particles(0, phx.DOMAIN, _particles(rng, dim, 6000, nc, [0] * dim, h, source))
    g = phx.Level(dim, order, fn, h, lower=flo, apply_tuning_table=False)
    o = O.Sim(dim, order, fn, h, lower=flo)
    for k in range(6):
        a = 0.02 * rng.standard_normal(g.shape(phx.F_EAVG + k)) + (0.3 if k == 4 else 0.0)
        g.set(phx.F_EAVG + k, a)
        o.set(O.F_EAVG + k, a)
    ghosts = [(tuple([flo[0] - 2] + flo[1:]), tuple([flo[0] - 1] + fhi[1:]))]
    own = _particles(rng, dim, 5000, fn, flo, h, 1.0)
    if into == "ghosts-first":
        g.refine_particles(coarse, ghosts, kind=phx.LEVEL_GHOST)
    g.set_particles(0, phx.DOMAIN, own)
    if into == "domain":
        g.refine_particles(coarse, [(tuple(flo), tuple(fhi))], kind=phx.DOMAIN)
    g.sort_particles()
    if into == "ghosts":
        g.refine_particles(coarse, ghosts, kind=phx.LEVEL_GHOST)
    for kind, okind in ((phx.DOMAIN, 0), (phx.LEVEL_GHOST, 2)):
        p = g.get_particles(0, kind)
        assert kind == phx.DOMAIN or into == "domain" or len(p["weight"]) > 50
        o.set_particles(0, okind, p)
    for step, mode in enumerate(4 * [phx.MODE_DOMAIN_ONLY, phx.MODE_ALL]):
        if step == 4:
            g.sort_particles()  # what entered the domain is now in its segments
        g.update_populations(DT, mode)
        o.update_populations(DT, mode)
        for k in range(5):
            U.assert_close(g.get(phx.f_pop(0, k)), o.get(O.f_pop(0, k)), what=f"mode {mode} moment {k}")
        for kind, okind in ((phx.DOMAIN, 0), (phx.PATCH_GHOST, 1), (phx.LEVEL_GHOST, 2)):
            U.assert_same_particles(g.get_particles(0, kind), o.get_particles(0, okind), what=f"kind {kind}")
    g.close()
    coarse.close()
