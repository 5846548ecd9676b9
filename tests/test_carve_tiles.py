"""Hull carving by image tiles (k_hull.hip: k_carve_cut, k_carve_tiles) against one walk per history and method, which
shares no code with it beyond the voxel formulas: the counts are integers and equal (hull_detection, DS.cu:6607;
SC_GPU :6681, MSC_GPU :6799, SM_GPU :6997).  PCT_CARVE_TILES selects the path: the rule takes tiles from 2^18
histories on.
"""
from __future__ import annotations

import numpy as np
import pytest

from cases import small_cylinder, small_head

pytestmark = pytest.mark.gpu

KINDS = ("sc_hull", "msc_counts", "sm_counts")


def _counts(monkeypatch, P, data, **env):
    from pct_reconstruction_amd import Reconstruction
    for k in ("PCT_CARVE_TILES", "PCT_CARVE_TABLE"):
        monkeypatch.delenv(k, raising=False)
    for k, v in env.items():
        monkeypatch.setenv(k, v)
    with Reconstruction(P) as r:
        r.load_histories(data["t"], data["v"], data["u"], data["wepl"], data["angle_deg"])
        r.import_and_process_data()
        out = {k: r.image(k).reshape(-1) for k in KINDS}
        print(f"[carve {env}] {r.count('recon_volume')} histories, most visits {out['sm_counts'].max()}", flush=True)
        return out


# grids below a tile, of a whole tile, one voxel past it and of several with remainders; odd slice counts and one
# slice; histories from none to the rule's own path, with paths along an axis (no slope in z, x or y)
@pytest.mark.parametrize("make, n, kw", [
    (small_head, 30000, dict(columns=50, rows=37, slice_thickness=0.7)),
    (small_head, 30000, dict(columns=64, rows=64, slice_thickness=0.4)),
    (small_head, 30000, dict(columns=65, rows=129, slice_thickness=0.3)),
    (small_head, 20000, dict(columns=200, rows=256, slice_thickness=0.25)),
    (small_cylinder, 30000, dict(columns=16, rows=16, slice_thickness=2.5)),
    (small_cylinder, 30000, dict(columns=128, rows=127, slice_thickness=5.0)),
    (small_cylinder, 400, dict(columns=130, rows=70, slice_thickness=1.0)),
    (small_head, 300000, dict(columns=96, rows=64, slice_thickness=0.4)),
])
@pytest.mark.parametrize("axes", [False, True])
def test_tiles_count_as_single_walks(monkeypatch, make, n, kw, axes):
    P, data = make(n=n, seed=71, **dict(kw, sc_on=1, msc_on=1, sm_on=1))
    if axes:
        k = np.arange(data["wepl"].size)
        data = {key: np.array(val) for key, val in data.items()}
        data["v"][:, k % 3 == 0] = data["v"][0, k % 3 == 0]  # no slope in z
        data["t"][:, k % 2 == 0] = data["t"][0, k % 2 == 0]  # along x or y at these angles
        data["angle_deg"][k % 2 == 0] = 90.0 * (k[k % 2 == 0] // 2 % 4)
    by_walks = _counts(monkeypatch, P, data, PCT_CARVE_TABLE="0")
    by_tiles = _counts(monkeypatch, P, data, **({} if n >= 1 << 18 else {"PCT_CARVE_TILES": "1"}))
    assert by_walks["sm_counts"].max() > 1
    for k in KINDS:
        assert np.array_equal(by_walks[k], by_tiles[k]), k
