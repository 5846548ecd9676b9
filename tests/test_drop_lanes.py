"""The row kernel's lanes per history, by rule and as set (k_drop2.hip: row_lanes), give the same image bit for bit:
a row is regrouped only where no partial sum rounds (DS.cu:9245)."""
from __future__ import annotations

import numpy as np
import pytest

from cases import small_cylinder

pytestmark = pytest.mark.gpu


# lists about and above 128 entries in small blocks (32 lanes by rule), short lists (16), and blocks above the rule's
# size
@pytest.mark.parametrize("kw", [dict(columns=256, rows=256, drop_block_size=640), dict(columns=200, rows=180),
                                dict(columns=64, rows=64), dict(columns=256, rows=256, drop_block_size=9000)])
def test_lanes_by_rule_match_every_setting(monkeypatch, kw):
    from pct_reconstruction_amd import Reconstruction
    P, data = small_cylinder(n=30000, seed=23, **kw)
    out = []
    for lanes in (None, 16, 32, 64):
        with Reconstruction(P) as r:
            if lanes:
                r.set_launch(drop_row_lanes=lanes)
            r.load_histories(data["t"], data["v"], data["u"], data["wepl"], data["angle_deg"])
            r.preprocessing()
            r.reconstruction_cuts()
            r.build_mlp_lists()
            r.DROP(2)
            c = r.metrics()["counts"]
            print(f"[lanes {lanes}] {c['list_entries'] / c['reconstruction']:.0f} entries a list", flush=True)
            out.append(r.image("x").reshape(-1))
    for x in out[1:]:
        assert np.array_equal(out[0], x)
