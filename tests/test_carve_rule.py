"""The rule by which the hull counts go by image tiles (k_hull.hip: carve_tiles_worth): not on grids that are coarse for
the number of histories, where the hash table is faster.  The counts are those of the other path (hull_detection,
DS.cu:6607)."""
from __future__ import annotations

import numpy as np
import pytest

from cases import small_head

pytestmark = pytest.mark.gpu


# histories per voxel from 1 to 60; one method on a small grid, and both
@pytest.mark.parametrize("n, kw, tiles", [
    (400000, dict(columns=96, rows=64, slice_thickness=0.4), True),
    (400000, dict(columns=64, rows=64, slice_thickness=0.4), True),
    (400000, dict(columns=64, rows=64, slice_thickness=0.4, msc_on=0, hull_type=3), False),
    (400000, dict(columns=120, rows=100, slice_thickness=0.4, msc_on=0, hull_type=3), True),
    (400000, dict(columns=64, rows=64, slice_thickness=1.0), False),
    (400000, dict(columns=33, rows=31, slice_thickness=1.2), False),
    (1500000, dict(columns=90, rows=70, slice_thickness=0.4), False),
])
def test_the_rule_for_tiles_of_the_carve(monkeypatch, n, kw, tiles):
    from pct_reconstruction_amd import Reconstruction
    P, data = small_head(n=n, seed=71, **kw)
    kinds = [k for k, on in (("msc_counts", P.msc_on), ("sm_counts", P.sm_on)) if on]
    out = []
    for setting in (None, "0" if tiles else "1"):
        if setting:
            monkeypatch.setenv("PCT_CARVE_TILES", setting)
        with Reconstruction(P) as r:
            r.load_histories(data["t"], data["v"], data["u"], data["wepl"], data["angle_deg"])
            r.import_and_process_data()
            path, kept = r.metrics()["carve"], r.count("recon_volume")
            assert kept >= 1 << 18
            assert path["by_tiles"] == (kept if tiles == (setting is None) else 0)
            out.append([r.image(k) for k in kinds])
            print(f"[carve rule] {kw}: {kept / P.num_voxels:.1f} histories a voxel, {path}", flush=True)
    for a, b in zip(*out):
        assert np.array_equal(a, b)
