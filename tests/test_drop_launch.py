"""pct_set_launch: the row kernel's lanes can be left to the library's rule again (lanes 0, the default) after a fixed
number was set; the image is the same (k_drop2.hip: row_lanes)."""
from __future__ import annotations

import inspect

import numpy as np
import pytest

from cases import small_cylinder


def test_the_defaults_leave_the_lanes_to_the_rule():
    from pct_reconstruction_amd import Reconstruction
    assert inspect.signature(Reconstruction.set_launch).parameters["drop_row_lanes"].default == 0


@pytest.mark.gpu
def test_lanes_by_rule_again_after_a_fixed_number():
    from pct_reconstruction_amd import Reconstruction
    P, data = small_cylinder(n=20000, seed=23, columns=256, rows=256, drop_block_size=640)
    with Reconstruction(P) as r:
        assert r.metrics()["drop_plan"]["row_lanes"] == 0
        r.load_histories(data["t"], data["v"], data["u"], data["wepl"], data["angle_deg"])
        r.preprocessing()
        r.reconstruction_cuts()
        r.build_mlp_lists()
        out = []
        for kw, lanes in ((dict(), 0), (dict(drop_row_lanes=64), 64), (dict(), 0), (dict(drop_row_lanes=16), 16),
                          (dict(drop_row_lanes=0, drop_col_voxels=2), 0)):
            r.set_launch(**kw)
            assert r.metrics()["drop_plan"]["row_lanes"] == lanes
            r.reset_iterate()
            r.DROP(2)
            out.append(r.image("x"))
        for bad in (-1, 3, 128):
            with pytest.raises(RuntimeError):
                r.set_launch(drop_row_lanes=bad)
    for x in out[1:]:
        assert np.array_equal(out[0], x)
