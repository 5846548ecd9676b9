"""List segments of which some take a plan over image tiles and some the sorted lists (the rule of
pct_tiles_prepare: 2^25 list slots): every DROP iteration walks all of them (segments.hip; the reference's
partial-transfer DROP, DS.cu:9590-9742), so both plans' buffers stay from one to the next.
"""
from __future__ import annotations

import numpy as np
import pytest

from cases import small_cylinder

pytestmark = pytest.mark.gpu


def test_segments_of_both_plans_keep_their_buffers():
    from pct_reconstruction_amd import Reconstruction
    P, data = small_cylinder(n=420000, seed=17, columns=200, rows=200, slice_thickness=0.25, drop_block_size=40000,
                             histories_per_block=320)
    out = []
    for segment in (0, 5 * 40000):
        Q = P.copy()
        Q.list_segment_histories = segment
        with Reconstruction(Q) as r:
            r.load_histories(data["t"], data["v"], data["u"], data["wepl"], data["angle_deg"])
            r.preprocessing()
            r.reconstruction_cuts()
            r.build_mlp_lists()
            n = r.count("reconstruction")
            r.DROP(1)
            first = r.metrics()
            r.DROP(2)
            last = r.metrics()
            out.append(r.image("x"))
            print(f"[segment plans] {n} histories, segment {segment}: {last['counts']}, {last['drop_plan']}", flush=True)
            if segment:
                assert n % segment and n > segment
                assert last["counts"]["list_slots"] < 1 << 25  # the last segment's: by the sorted lists
                assert not last["drop_plan"]["tiles"]
                assert last["counts"]["device_allocations"] == first["counts"]["device_allocations"]
            else:
                assert last["drop_plan"]["tiles"]
    assert np.array_equal(out[0], out[1])
