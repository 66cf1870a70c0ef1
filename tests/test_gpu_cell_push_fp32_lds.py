"""The mixed-precision cell-grouped push where its tile and stage do not fit in LDS (3D order 3 with
segments of 1x1x64 cells): every particle is pushed by itself and deposits straight into the moment
arrays. The run says so once on stderr; moments within 1e-5 of the FP64 oracle, the bound of the family's
other one-step tests."""
import numpy as np
import pytest

import oracle_lib as O
import parity_util as U
from phare_amd import phx
from phare_amd import workloads as W

pytestmark = pytest.mark.gpu


def test_fp32_tile_beyond_lds(capfd):
    print("[gpu] FP32 cell push beyond LDS", flush=True)
    wl = W.uniform3d(ncells=(10, 10, 64), ppc=4, order=3)
    g = phx.Level(3, 3, wl.ncells, wl.dx, masses=wl.masses, Te=wl.Te, capacity=wl.n_particles,
                  precision=phx.PRECISION_FP32, apply_tuning_table=False)
    g.set_tuning(segment_shape=[1, 1, 64], sort_interval=1)
    o = O.Sim(3, 3, wl.ncells, wl.dx, masses=wl.masses, Te=wl.Te)
    wl.setup(g, phx.F_B)
    wl.setup(o, O.F_B)
    g.advance(wl.dt, 1)
    o.advance(wl.dt, 1)
    g.sync()
    assert capfd.readouterr().err.count("does not fit for segments of 1x1x64 cells") == 1
    for k in range(5):
        U.assert_close(g.get(phx.f_pop(0, k)), o.get(O.f_pop(0, k)), 1e-5, what=f"moment {k}")
    assert g.diagnostics()["count"] == o.diagnostics()["count"]
    g.close()
