"""Hull carving by image tiles in several batches, and with the last histories counted by the hash table
(k_hull.hip: carve_by_tiles, k_carve_all), against one walk per history and method: the counts are integers and equal
(hull_detection, DS.cu:6607).  The metrics say how many histories each path counted."""
from __future__ import annotations

import numpy as np
import pytest

from cases import small_head

pytestmark = pytest.mark.gpu

KINDS = ("sc_hull", "msc_counts", "sm_counts")


def _counts(monkeypatch, P, data, **env):
    from pct_reconstruction_amd import Reconstruction
    for k in ("PCT_CARVE_TILES", "PCT_CARVE_TABLE", "PCT_CARVE_BATCH", "PCT_CARVE_BATCHES"):
        monkeypatch.delenv(k, raising=False)
    for k, v in env.items():
        monkeypatch.setenv(k, str(v))
    with Reconstruction(P) as r:
        r.load_histories(data["t"], data["v"], data["u"], data["wepl"], data["angle_deg"])
        for _ in range(2):  # the second run finds the scratch of the first
            r.import_and_process_data()
        return {k: r.image(k).reshape(-1) for k in KINDS}, r.count("recon_volume"), r.metrics()["carve"]


# batches of a size that leaves a remainder, of one history less than all, and of all; none to all of them by tiles
@pytest.mark.parametrize("batch, batches", [(7001, -1), (7001, 2), (7001, 0), ("n-1", -1), ("n-1", 1), ("n", 1), (1 << 20, -1)])
def test_batches_count_as_single_walks(monkeypatch, batch, batches):
    P, data = small_head(n=30000, seed=73, columns=70, rows=130, slice_thickness=0.3, sc_on=1)  # odd numbers of tiles
    by_walks, n, path = _counts(monkeypatch, P, data, PCT_CARVE_TABLE=0)
    assert path == dict(by_tiles=0, tile_batches=0, by_walks=n)
    batch = {"n": n, "n-1": n - 1}.get(batch, batch)
    by_tiles, _, path = _counts(monkeypatch, P, data, PCT_CARVE_TILES=1, PCT_CARVE_BATCH=batch, PCT_CARVE_BATCHES=batches)
    all_batches = -(-n // batch)
    done = all_batches if batches < 0 else min(batches, all_batches)
    print(f"[carve] {n} histories, {path}", flush=True)
    assert path == dict(by_tiles=min(done * batch, n), tile_batches=done, by_walks=n - min(done * batch, n))
    for k in KINDS:
        assert np.array_equal(by_walks[k], by_tiles[k]), k


def test_the_rule_takes_tiles_from_a_quarter_million_histories(monkeypatch):
    P, data = small_head(n=300000, seed=71, columns=96, rows=64, slice_thickness=0.4, sc_on=1)
    _, n, path = _counts(monkeypatch, P, data)
    assert n >= 1 << 18 and path == dict(by_tiles=n, tile_batches=1, by_walks=0)
    P, data = small_head(n=200000, seed=71, columns=96, rows=64, slice_thickness=0.4, sc_on=1)
    _, n, path = _counts(monkeypatch, P, data)
    assert path == dict(by_tiles=0, tile_batches=0, by_walks=n)
