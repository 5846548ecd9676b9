"""DROP over image tiles (k_drop_tiles.hip) against the sorted lists (k_drop2.hip), bit for bit: the same updates
summed in the same order per voxel, and row sums regrouped only where no partial sum can round
(DROP_full_tx_iteration, DS.cu:9537-9589).  PCT_DROP_TILES selects the path: the rule takes tiles only for plans
of 2^25 list slots and more (the full-size tests run them by the rule).
"""
from __future__ import annotations

import numpy as np
import pytest

from cases import small_cylinder, small_head

pytestmark = pytest.mark.gpu


def _run(monkeypatch, tiles, P, data, iterations, x=None, group_entries=None):
    from pct_reconstruction_amd import Reconstruction
    monkeypatch.setenv("PCT_DROP_TILES", str(tiles))
    if group_entries is not None:
        monkeypatch.setenv("PCT_DROP_GROUP_ENTRIES", str(group_entries))
    with Reconstruction(P) as r:
        r.load_histories(data["t"], data["v"], data["u"], data["wepl"], data["angle_deg"])
        r.preprocessing()
        r.reconstruction_cuts()
        r.build_mlp_lists()
        if x is not None:
            r.set_image(x)
        r.DROP(1)
        first, plan = r.image("x").reshape(-1), r.metrics()["drop_plan"]
        r.DROP(iterations - 1)
        prof = r.profile_drop(1)
        return dict(first=first, x=r.image("x").reshape(-1), residual=r.residual(), plan=plan, prof=prof,
                    n=r.count("reconstruction"))


def _compare(monkeypatch, P, data, iterations, taken=True, **kw):
    a = _run(monkeypatch, 0, P, data, iterations, **kw)
    b = _run(monkeypatch, 1, P, data, iterations, **kw)
    print(f"[tiles] {a['n']} histories, {a['prof']['blocks']} blocks, {a['prof']['summed']} entries, "
          f"{a['prof']['touched']} touched voxels; tiles {b['plan']['tiles']}", flush=True)
    assert not a["plan"]["tiles"] and b["plan"]["tiles"] == taken
    assert np.array_equal(a["first"], b["first"])
    assert np.array_equal(a["x"], b["x"])
    assert abs(a["residual"] - b["residual"]) <= 1e-12 * a["residual"]  # the same squares in the same order
    for k in ("blocks", "histories", "gathered", "summed", "touched"):
        assert a["prof"][k] == b["prof"][k], k
    return b


# grids with a partial last tile in every direction, one voxel past a tile, and odd slice counts; blocks from one
# that leaves histories unprocessed in every block (quirk A3) to one for all histories
@pytest.mark.parametrize("make, kw", [
    (small_head, dict(columns=50, rows=37, slice_thickness=0.7, drop_block_size=6400, histories_per_block=640)),
    (small_head, dict(columns=17, rows=33, slice_thickness=1.0, drop_block_size=2400, histories_per_block=700,
                      min_mlp_length=5)),
    (small_cylinder, dict(columns=64, rows=64, slice_thickness=2.5, drop_block_size=1500, histories_per_block=1)),
    (small_cylinder, dict(columns=64, rows=64, slice_thickness=0.4, drop_block_size=60000, histories_per_block=1)),
    (small_cylinder, dict(columns=16, rows=16, slice_thickness=1.0, drop_block_size=200, histories_per_block=1,
                          min_mlp_length=5)),
    (small_head, dict(columns=120, rows=96, slice_thickness=0.33, drop_block_size=3200, histories_per_block=320)),
])
@pytest.mark.parametrize("accum", [0, 1, 2])
def test_tiles_match_the_sorted_lists(monkeypatch, make, kw, accum):
    P, data = make(n=40000, seed=61, drop_accum=accum, **kw)
    b = _compare(monkeypatch, P, data, 3)
    assert b["prof"]["summed"] > 0


@pytest.mark.parametrize("group_entries", [1, 400000])
def test_tiles_in_many_groups(monkeypatch, group_entries):
    """Blocks transposed in groups: consecutive blocks' lists lie in different groups' arrays."""
    P, data = small_head(n=50000, seed=53, drop_block_size=3200, histories_per_block=700)
    _compare(monkeypatch, P, data, 2, group_entries=group_entries)


def test_tiles_with_short_paths_and_empty_blocks(monkeypatch):
    """Blocks of 7 histories with MIN_MLP_LENGTH 55: blocks, and with groups of one block groups, without a segment."""
    P, data = small_cylinder(n=6000, seed=8, drop_block_size=7, histories_per_block=1, min_mlp_length=55)
    _compare(monkeypatch, P, data, 2)
    _compare(monkeypatch, P, data, 2, group_entries=1)


def test_tiles_with_untabulated_paths(monkeypatch):
    P, data = small_head(n=30000, seed=29, mlp_algorithm=0)
    _compare(monkeypatch, P, data, 2)


def test_tiles_too_full_fall_back(monkeypatch):
    """A block of 60000 histories on 16 x 16 voxels passes more than 1022 segments through a tile."""
    P, data = small_cylinder(n=60000, seed=11, columns=16, rows=16, slice_thickness=4.0, drop_block_size=60000,
                             histories_per_block=1, min_mlp_length=5)
    _compare(monkeypatch, P, data, 2, taken=False)


def test_tiles_without_a_long_path(monkeypatch):
    P, data = small_cylinder(n=6000, seed=8, min_mlp_length=500)
    _compare(monkeypatch, P, data, 2, taken=False)


@pytest.mark.parametrize("values", ["ordered", "nan", "zeros", "denormal"])
def test_row_sums_that_round_in_tiles(monkeypatch, oracle, values):
    """Images whose row sums depend on the order, hold a NaN and an infinity, are all zero, or subnormal: rows
    fall back to the sum in list order, as in the oracle (DS.cu:9245)."""
    P, data = small_cylinder(n=30000, seed=12)
    k = np.arange(P.num_voxels)
    x = np.where(k % 3 == 0, 1.0, 2.0 ** -53).astype(np.float32)
    if values == "nan":
        x[P.num_voxels // 2 + 20] = np.nan
        x[P.num_voxels // 2 + 90] = np.inf
    elif values == "zeros":
        x[:] = 0
    elif values == "denormal":
        x = (x * np.float32(2.0 ** -100)).astype(np.float32)
    from pct_reconstruction_amd import Reconstruction
    out = []
    for tiles in (0, 1):
        monkeypatch.setenv("PCT_DROP_TILES", str(tiles))
        with Reconstruction(P) as r:
            r.load_histories(data["t"], data["v"], data["u"], data["wepl"], data["angle_deg"])
            r.preprocessing()
            r.reconstruction_cuts()
            r.build_mlp_lists()
            r.set_image(x)
            r.DROP(2)
            assert r.metrics()["drop_plan"]["tiles"] == bool(tiles)
            out.append(r.image("x").reshape(-1))
    assert np.array_equal(out[0], out[1], equal_nan=True)
    if values == "ordered":
        ref = oracle.run_pipeline(P, data, stop_after="lists")
        x_ref = x
        for _ in range(2):
            x_ref = oracle.drop_iteration(P, ref["offsets"], ref["voxels"], ref["chord"], ref["wepl_recon"], x_ref,
                                          accum=P.drop_accum)
        assert np.array_equal(out[1], x_ref)


def test_tiles_inside_segments_and_with_tvs(monkeypatch):
    """Segments of whole blocks rebuild the tiles' plan; TVS works on the linear image between iterations."""
    P, data = small_cylinder(n=60000, seed=41, drop_block_size=3200, histories_per_block=320, tvs_on=1)
    from pct_reconstruction_amd import Reconstruction
    out = []
    for tiles, seg in ((0, 0), (1, 0), (1, 9600)):
        monkeypatch.setenv("PCT_DROP_TILES", str(tiles))
        Q = P.copy()
        Q.list_segment_histories = seg
        with Reconstruction(Q) as r:
            r.load_histories(data["t"], data["v"], data["u"], data["wepl"], data["angle_deg"])
            r.preprocessing()
            r.reconstruction_cuts()
            r.build_mlp_lists()
            r.DROP(3)
            out.append((r.image("x"), r.residual()))
    for x, res in out[1:]:
        assert np.array_equal(x, out[0][0])
        assert abs(res - out[0][1]) <= 1e-12 * out[0][1]


def test_tiles_on_imported_lists_with_repeated_voxels(monkeypatch, tmp_path):
    """Imported path lists may jump between tiles and visit a voxel again, also within one tile: the repeated visit
    adds its update again, as in the reference's list walk (DS.cu:9522-9536)."""
    from pct_reconstruction_amd import Reconstruction
    P, data = small_cylinder(n=20000, seed=9, iterations=1)
    with Reconstruction(P) as r:
        r.load_histories(data["t"], data["v"], data["u"], data["wepl"], data["angle_deg"])
        r.preprocessing()
        r.reconstruction_cuts()
        r.build_mlp_lists()
        off, vox = r.lists()
        r.export_preprocessed(tmp_path)
    rng = np.random.default_rng(3)
    vox = vox.copy()
    n = off.size - 1
    for i in rng.choice(n, 300, replace=False):
        a, b = off[i], off[i + 1]
        if b - a > 6:
            vox[a + 4] = vox[a + 2]              # A B A within a tile
            vox[a + 5] = rng.integers(P.num_voxels)  # a jump
    (np.concatenate([np.array([n], np.uint32), vox])).tofile(tmp_path / "MLP.bin")
    out = []
    for tiles in (0, 1):
        monkeypatch.setenv("PCT_DROP_TILES", str(tiles))
        with Reconstruction(P) as r:
            r.import_preprocessed(tmp_path)
            r.DROP(2)
            assert r.metrics()["drop_plan"]["tiles"] == bool(tiles)
            out.append((r.image("x"), r.residual()))
    assert np.array_equal(out[0][0], out[1][0])
    assert abs(out[0][1] - out[1][1]) <= 1e-12 * out[0][1]


@pytest.mark.parametrize("kw", [dict(), dict(columns=150, rows=150, slice_thickness=0.5)])
@pytest.mark.parametrize("every", [37, 2500])
def test_some_rows_round_in_tiles(monkeypatch, kw, every):
    """Tiles with a few tiny values: their segments bound their own values, the rows through a tiny one are summed in
    list order by a whole wavefront (also past 256 entries), the others as they are; bit for bit the sorted lists."""
    P, data = small_head(n=30000, seed=19, drop_block_size=6000, histories_per_block=640, **kw)
    rng = np.random.default_rng(4)
    x = (1.0 + 0.3 * rng.standard_normal(P.num_voxels)).astype(np.float32)
    x[::every] *= np.float32(1e-12)
    b = _compare(monkeypatch, P, data, 3, x=x)
    assert b["prof"]["summed"] > 0
