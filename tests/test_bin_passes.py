"""The bin passes (k_preproc.hip: k_bin_offsets, k_bin_stats, k_compact) against the oracle where a wavefront's 64 bins
hold from no history to many times what its LDS stages at once (kStatChunk): binning (DS.cu:5518-5546), means and
deviations (:5644-5737), the cuts (:5937-5971) and the histories that are left, value by value."""
from __future__ import annotations

import numpy as np
import pytest

from cases import small_cylinder, small_head
from test_gpu_parity import H_NAMES

pytestmark = pytest.mark.gpu


# about 1, 17, 300 and 4000 histories to a bin; a handful of histories; both readings of bin 0's quirk
@pytest.mark.parametrize("make, n, kw", [
    (small_head, 40000, dict(t_bin_size=0.5, v_bin_size=1.0, angular_bin_size=8.0)),
    (small_head, 40000, dict(t_bin_size=2.0, v_bin_size=4.0, angular_bin_size=12.0)),
    (small_cylinder, 40000, dict(t_bin_size=12.0, v_bin_size=4.5, angular_bin_size=40.0)),
    (small_cylinder, 40000, dict(t_bin_size=35.0, v_bin_size=9.0, angular_bin_size=45.0)),
    (small_cylinder, 65, dict(t_bin_size=0.5, v_bin_size=1.0, angular_bin_size=8.0)),
])
@pytest.mark.parametrize("quirk", [0, 1])
def test_bins_match_the_oracle(oracle, make, n, kw, quirk):
    from pct_reconstruction_amd import Reconstruction
    P, data = make(n=n, seed=83, quirk_a1_bin0=quirk, **kw)
    ref = oracle.run_pipeline(P, data, stop_after="cuts")
    with Reconstruction(P) as r:
        r.load_histories(data["t"], data["v"], data["u"], data["wepl"], data["angle_deg"])
        r.import_and_process_data()
        r.hull_detection_finish()
        r.statistical_calculations_and_cuts()
        pre, post = r.bins("counts_pre"), r.bins("counts_post")
        print(f"[bins] {pre.size} bins, most in one {pre.max()}, {r.count('post_cuts')} histories left", flush=True)
        assert np.array_equal(pre, ref["counts_pre"])
        for k, name in enumerate(("wepl", "ut", "uv")):
            assert np.array_equal(r.bins("mean_" + name), ref["mean"][k], equal_nan=True), name
            assert np.array_equal(r.bins("std_" + name), ref["std"][k], equal_nan=True), name
        assert np.array_equal(post, ref["counts_post"])
        assert np.array_equal(r.bins("sinogram"), ref["sinogram_sum"])
        assert r.count("post_cuts") == ref["h_cut"].shape[1]
        for k, name in enumerate(H_NAMES):
            assert np.array_equal(r.histories(name), ref["h_cut"][k]), name
