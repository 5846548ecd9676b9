"""A context that reconstructs again finds its buffers: no device memory is allocated from the second run on, with the
hull counts by image tiles (k_hull.hip: carve_by_tiles) and by the hash table, with image tiles and sorted lists for
DROP, and the images are the same."""
from __future__ import annotations

import numpy as np
import pytest

from cases import small_cylinder, small_head

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("make, n, kw", [
    (small_head, 400000, dict(columns=96, rows=96, slice_thickness=0.4)),
    (small_cylinder, 30000, dict()),
    (small_cylinder, 420000, dict(columns=200, rows=200, slice_thickness=0.25, drop_block_size=40000, msc_on=1)),
])
def test_a_second_run_allocates_nothing(make, n, kw):
    from pct_reconstruction_amd import Reconstruction
    P, data = make(n=n, seed=37, **kw)
    with Reconstruction(P) as r:
        r.load_histories(data["t"], data["v"], data["u"], data["wepl"], data["angle_deg"])
        images, made = [], []
        for _ in range(3):
            images.append(r.run())
            m = r.metrics()
            made.append(m["counts"]["device_allocations"])
        print(f"[buffers] allocations {made}, {m['carve']}, {m['drop_plan']}", flush=True)
        assert made[0] < 250 and made[2] == made[1] == made[0]
    assert np.array_equal(images[0], images[1]) and np.array_equal(images[0], images[2])
