"""The autotuner can make every entry of the committed table again (phare_amd/autotune.py): the entry's name
gives its workload, and the settings it holds besides the defaults are ones that the tuner searches there."""
import json

import pytest

from phare_amd import autotune

# defaults of include/phx.h that the entries may carry along
DEFAULTS = {2: dict(segment_shape=[2, 32, 1], rows_per_item=32, tile_row_pad=16, sort_interval=30, tile_copies=8,
                    deposit_window=0)}


@pytest.mark.parametrize("entry", json.load(open(autotune.TABLE)), ids=lambda e: f"{e['workload']}-{e['precision']}")
def test_entry_can_be_made_again(entry):
    wl = autotune.workload(entry["workload"])
    assert autotune.name_of(wl) == entry["workload"]
    assert (wl.dim, wl.order, wl.ppc) == (entry["dim"], entry["order"], entry["ppc"])
    searched = autotune.space(wl.dim, wl.order, entry["precision"])
    changed = {k: v for k, v in entry["tuning"].items() if v != DEFAULTS[wl.dim][k]}
    assert changed, "an entry of the defaults"
    for k, v in changed.items():
        assert v in searched[k], (k, v)


def test_names():
    wl = autotune.workload("harris2d-o3-n190x150-p64")
    assert wl.ncells == [190, 150] and wl.order == 3 and wl.ppc == 64
    assert autotune.workload("uniform3d-n12").ncells == [12, 12, 12]
    assert autotune.workload("uniform1d-n64-p16").ncells == [64]
    for bad in ("harris3d", "harris2d-x4", "harris2d-n8x8x8", "harris2d-o"):
        with pytest.raises(SystemExit):
            autotune.workload(bad)


def test_only_settings_that_act_are_searched():
    assert "tile_row_pad" not in autotune.space(2, 2, "fp64") and "tile_row_pad" in autotune.space(2, 2, "fp32")
    assert "deposit_window" not in autotune.space(2, 3, "fp32") and "deposit_window" in autotune.space(1, 1, "fp32")
    assert 7 in autotune.space(3, 2, "fp32")["sort_interval"]
