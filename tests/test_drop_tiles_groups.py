"""Transposition groups without a segment in a plan over image tiles (k_drop_tiles.hip: build_group): a group whose
paths are all shorter than MIN_MLP_LENGTH, in a context whose earlier plan had segments there.  Its rows say that the
histories have none, and DROP and the residual equal those of the sorted lists bit for bit (k_drop2.hip;
DROP_full_tx_iteration, DS.cu:9537-9589).
"""
from __future__ import annotations

import shutil

import numpy as np
import pytest

from cases import small_cylinder

pytestmark = pytest.mark.gpu

BLOCK = 1500


def _cut_paths(off, vox, path, short_blocks):
    """The exported lists with the paths of some DROP blocks cut to 7 voxels."""
    n = off.size - 1
    cnt = np.diff(off)
    short = np.isin(np.arange(n) // BLOCK, short_blocks)
    cnt[short] = np.minimum(cnt[short], 7)
    keep = np.arange(vox.size) - np.repeat(off[:-1], np.diff(off)) < np.repeat(cnt, np.diff(off))
    np.concatenate([np.array([n], np.uint32), vox[keep]]).astype(np.uint32).tofile(path / "MLP.bin")
    np.concatenate([np.array([n], np.uint32), cnt.astype(np.uint32)]).tofile(path / "voxels_per_path.bin")


# the first, the last, two in the middle, and all but one of the groups
@pytest.mark.parametrize("which", ["first", "last", "middle", "all_but_one"])
def test_groups_without_segments_after_a_plan_with_them(monkeypatch, tmp_path, which):
    from pct_reconstruction_amd import Reconstruction
    P, data = small_cylinder(n=20000, seed=9, drop_block_size=BLOCK, histories_per_block=1)
    full, cut = tmp_path / "full", tmp_path / "cut"
    with Reconstruction(P) as r:
        r.load_histories(data["t"], data["v"], data["u"], data["wepl"], data["angle_deg"])
        r.preprocessing()
        r.reconstruction_cuts()
        r.build_mlp_lists()
        off, vox = r.lists()
        r.export_preprocessed(full)
    blocks = -(-(off.size - 1) // BLOCK)
    assert blocks >= 4
    shutil.copytree(full, cut)
    _cut_paths(off, vox, cut, {"first": [0], "last": [blocks - 1], "middle": [1, 2],
                               "all_but_one": [b for b in range(blocks) if b != 2]}[which])
    out = []
    for tiles in (0, 1):
        monkeypatch.setenv("PCT_DROP_TILES", str(tiles))
        monkeypatch.setenv("PCT_DROP_GROUP_ENTRIES", "1")  # a group per block
        with Reconstruction(P) as r:
            r.import_preprocessed(full)
            r.DROP(1)
            r.import_preprocessed(cut)
            r.DROP(2)
            assert r.metrics()["drop_plan"]["tiles"] == bool(tiles)
            prof = r.profile_drop(1)
            out.append((r.image("x"), r.residual(), prof))
            print(f"[groups {which}] tiles {tiles}: {blocks} blocks, {prof['summed']} entries", flush=True)
    assert out[0][2]["summed"] > 0
    assert np.array_equal(out[0][0], out[1][0])
    assert abs(out[0][1] - out[1][1]) <= 1e-12 * out[0][1]  # the same squares in the same order
    for k in ("blocks", "histories", "gathered", "summed", "touched"):
        assert out[0][2][k] == out[1][2][k], k
