"""The rule by which a DROP plan goes over image tiles (k_drop_tiles.hip: pct_tiles_prepare), on each of its sides: few or
crowded tiles and small blocks keep the sorted lists, before anything of the tiles' plan is allocated or built.  The
image is that of the sorted lists bit for bit (DROP_full_tx_iteration, DS.cu:9537-9589)."""
from __future__ import annotations

import numpy as np
import pytest

from cases import small_cylinder, small_head

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name, make, n, kw, tiles", [
    ("taken", small_cylinder, 420000, dict(columns=200, rows=200, slice_thickness=0.25, drop_block_size=40000), True),
    ("few tiles", small_head, 1100000, dict(columns=100, rows=100, slice_thickness=0.25, drop_block_size=20000), False),
    ("too many segments in a tile", small_cylinder, 700000, dict(columns=170, rows=170, slice_thickness=0.25,
                                                                 drop_block_size=60000), False),
    ("sparse tiles", small_cylinder, 420000, dict(columns=200, rows=200, slice_thickness=0.25, drop_block_size=3000),
     False),
    ("small blocks", small_cylinder, 900000, dict(columns=128, rows=128, slice_thickness=0.25, drop_block_size=5000),
     False),
])
def test_the_rule_for_tiles(monkeypatch, name, make, n, kw, tiles):
    from pct_reconstruction_amd import Reconstruction
    P, data = make(n=n, seed=3, histories_per_block=320, **kw)
    out, made = [], []
    for setting in ("0", "-1"):
        monkeypatch.setenv("PCT_DROP_TILES", setting)
        with Reconstruction(P) as r:
            r.load_histories(data["t"], data["v"], data["u"], data["wepl"], data["angle_deg"])
            r.preprocessing()
            r.reconstruction_cuts()
            before = r.metrics()["counts"]["device_allocations"]
            r.build_mlp_lists()
            m = r.metrics()
            made.append(m["counts"]["device_allocations"] - before)
            assert m["counts"]["list_slots"] >= 1 << 25  # smaller plans never ask the rule
            r.DROP(2)
            out.append(r.image("x"))
            print(f"[rule: {name}] {m['counts']['reconstruction']} histories, {m['counts']['list_slots']} slots, "
                  f"{made[-1]} allocations, {m['drop_plan']}", flush=True)
    assert m["drop_plan"]["tiles"] == tiles
    if not tiles:
        assert made[1] <= made[0] + 2  # the sample's counts
    assert np.array_equal(out[0], out[1])
