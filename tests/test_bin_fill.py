"""The bin statistics (k_preproc.hip: k_bin_stats) on both sides of the number of entries from which a wavefront's 64
bins are read from memory instead of through LDS (stat_staged), for few bins and for more than 2^17: means and
deviations (DS.cu:5644-5737), the cuts (:5937-5971) and the histories that are left, value by value against the oracle.
"""
from __future__ import annotations

import numpy as np
import pytest

from cases import small_head

pytestmark = pytest.mark.gpu

FINE = dict(t_bin_size=0.1, v_bin_size=0.25, angular_bin_size=4.0)
COARSE = dict(t_bin_size=2.0, v_bin_size=4.0, angular_bin_size=12.0)


# few bins, up to 2048 entries of 64 of them staged; one angle of many bins, up to 8192
@pytest.mark.parametrize("n, angles, bins, from_memory", [
    (30000, 0, COARSE, False), (60000, 0, COARSE, True), (150000, 1, FINE, False), (900000, 1, FINE, False),
    (1300000, 1, FINE, True)])
def test_bins_match_the_oracle_on_both_sides_of_the_rule(oracle, n, angles, bins, from_memory):
    from pct_reconstruction_amd import Reconstruction
    P, data = small_head(n=n, seed=89, **bins)
    if angles:
        data["angle_deg"] = np.full_like(data["angle_deg"], 40.0)
    ref = oracle.run_pipeline(P, data, stop_after="cuts")
    with Reconstruction(P) as r:
        r.load_histories(data["t"], data["v"], data["u"], data["wepl"], data["angle_deg"])
        r.import_and_process_data()
        r.hull_detection_finish()
        fill = np.bincount(r.histories("bin_num") // 64).max()
        r.statistical_calculations_and_cuts()
        print(f"[bin fill] {P.num_bins} bins, most in 64 of them {fill}, {r.count('post_cuts')} histories left", flush=True)
        assert (fill > (8192 if P.num_bins >= 1 << 17 else 2048)) == from_memory
        assert np.array_equal(r.bins("counts_pre"), ref["counts_pre"])
        for k, name in enumerate(("wepl", "ut", "uv")):
            assert np.array_equal(r.bins("mean_" + name), ref["mean"][k], equal_nan=True), name
            assert np.array_equal(r.bins("std_" + name), ref["std"][k], equal_nan=True), name
        assert np.array_equal(r.bins("counts_post"), ref["counts_post"])
        assert np.array_equal(r.bins("sinogram"), ref["sinogram_sum"])
        assert r.count("post_cuts") == ref["h_cut"].shape[1]
        assert np.array_equal(r.histories("x_entry"), ref["h_cut"][0])
