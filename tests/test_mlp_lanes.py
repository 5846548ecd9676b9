"""MLP lists by one, four or sixteen lanes per history (k_mlp.hip: mlp_lanes) are the same lists, entry by entry
(find_MLP_path_GPU_tabulated, DS.cu:9104-9262; find_MLP_path_GPU, :8895-9103)."""
from __future__ import annotations

import numpy as np
import pytest

from cases import small_cylinder, small_head

pytestmark = pytest.mark.gpu


# both list algorithms; lists of some hundred entries and of a few; image edges that cut paths (voxels past the last
# one are skipped); one history and enough for the rule's three choices
@pytest.mark.parametrize("make, n, kw", [
    (small_head, 30000, dict(columns=150, rows=130, slice_thickness=0.5)),
    (small_head, 30000, dict(mlp_algorithm=0)),
    (small_cylinder, 30000, dict(columns=16, rows=16, slice_thickness=2.5)),
    (small_cylinder, 30000, dict(mlp_algorithm=0, slice_thickness=4.0)),
    (small_cylinder, 80000, dict()),
    (small_cylinder, 260000, dict(mlp_algorithm=0)),
])
def test_lists_do_not_depend_on_the_lanes(monkeypatch, make, n, kw):
    from pct_reconstruction_amd import Reconstruction
    P, data = make(n=n, seed=31, **kw)
    out = []
    for lanes in ("0", "1", "4", "16"):
        monkeypatch.setenv("PCT_MLP_LANES", lanes)
        with Reconstruction(P) as r:
            r.load_histories(data["t"], data["v"], data["u"], data["wepl"], data["angle_deg"])
            r.preprocessing()
            r.reconstruction_cuts()
            r.build_mlp_lists()
            off, vox = r.lists()
            out.append((off, vox, r.histories("chord"), r.histories("path_count")))
            print(f"[lanes {lanes}] {off.size - 1} histories, {vox.size} entries", flush=True)
    assert out[0][1].size > out[0][0].size
    for o in out[1:]:
        for a, b in zip(out[0], o):
            assert np.array_equal(a, b)
