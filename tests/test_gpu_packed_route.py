"""Which push the drop-in updater takes over an array that its compaction left packed, seen from the
velocities: the linear push gathers and accelerates in the reference's order of operations, the
cell-grouped one with fused multiply-adds, so that a level pushed by the linear kernel holds bit for bit
the velocities of an unsorted level with the same particles, and one pushed cell by cell does not (both
within 1e-12). A quarter of the particles outside their segments turns the array over to the linear push;
a call that ended in an error leaves no count behind."""
import numpy as np
import pytest

import oracle_lib as O
import parity_util as U
from phare_amd import phx

pytestmark = pytest.mark.gpu

CELLS = {2: (20, 37), 3: (12, 11, 13)}
DX = [0.3, 0.25, 0.2]
DT = 0.05


def _fields(dim):
    rng = np.random.default_rng(7)
    return lambda shape, k: 0.02 * rng.standard_normal(shape) + (0.3 if k == 4 else 0.0)


def _level(dim, order, p):
    g = phx.Level(dim, order, CELLS[dim], DX[:dim], apply_tuning_table=False)
    f = _fields(dim)
    for k in range(6):
        g.set(phx.F_EAVG + k, f(g.shape(phx.F_EAVG + k), k))
    g.set_particles(0, phx.DOMAIN, p)
    return g


def _particles(rng, dim, n):
    p = U.random_particles(rng, dim, n, CELLS[dim], [0] * dim, 0)
    # every direction between 0.04 and 0.1 cells per half step of DT
    p["v"] = rng.choice([-1.0, 1.0], (n, 3)) * rng.uniform(0.04, 0.1, (n, 3)) * np.array(DX) / (0.5 * DT)
    p["charge"] = np.ones(n)
    return p


def _next_push_is_linear(g, dim, order):
    """pushes g once more; whether it holds the velocities of the linear push bit for bit"""
    before = g.get_particles()
    same = _level(dim, order, before)
    o = O.Sim(dim, order, CELLS[dim], DX[:dim])
    f = _fields(dim)
    for k in range(6):
        o.set(O.F_EAVG + k, f(o.shape(O.F_EAVG + k), k))
    o.set_particles(0, 0, before)
    for sim in (g, same, o):
        sim.update_populations(DT, phx.MODE_ALL)
    a, b = U.sort_particles(g.get_particles()), U.sort_particles(same.get_particles())
    U.assert_same_particles(a, o.get_particles())
    U.assert_same_particles(b, o.get_particles())
    same.close()
    return np.array_equal(a["v"], b["v"])


@pytest.mark.parametrize("order", [1, 2, 3])
@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("appended,linear", [(0.02, False), (0.6, True)])
def test_a_quarter_outside_the_segments_ends_the_packed_push(appended, linear, dim, order):
    print(f"[gpu] packed route dim={dim} order={order} appended {appended}", flush=True)
    rng = np.random.default_rng(order)
    n = 30 * int(np.prod(CELLS[dim]))
    g = _level(dim, order, _particles(rng, dim, n))
    g.sort_particles()
    assert not _next_push_is_linear(g, dim, order)
    g.set_particles(0, phx.PATCH_GHOST, _particles(rng, dim, int(appended * n)))
    g.fill_ion_ghost_particles()
    assert not _next_push_is_linear(g, dim, order)  # this push counts them
    assert _next_push_is_linear(g, dim, order) == linear
    g.close()


@pytest.mark.parametrize("dim", [2, 3])
def test_a_failed_push_leaves_no_count(dim):
    print(f"[gpu] packed route after an error dim={dim}", flush=True)
    order = 2
    rng = np.random.default_rng(dim)
    g = _level(dim, order, _particles(rng, dim, 30 * int(np.prod(CELLS[dim]))))
    g.sort_particles()
    with pytest.raises(phx.PhxError):
        g.update_populations(100 * DT, phx.MODE_ALL)  # every particle moves more than two cells
    assert not _next_push_is_linear(g, dim, order)
    assert not _next_push_is_linear(g, dim, order)
    g.close()
