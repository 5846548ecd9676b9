"""FBP back-projection with eight voxels of a column per lane (k_fbp.hip: k_backproject, from 2^18 lanes on) against the
oracle, value by value, in both readings of the voxel decoding (backprojection_GPU2, DS.cu:6340-6479; :11124-11134).
Smaller grids take one voxel per lane; the parity tests run those."""
from __future__ import annotations

import numpy as np
import pytest

from cases import small_head

pytestmark = pytest.mark.gpu


# slices in whole groups of eight, one more, and seven in the last; a row length that is no multiple of a workgroup
@pytest.mark.parametrize("columns, rows, slices", [(512, 512, 8), (401, 330, 17), (256, 256, 31)])
@pytest.mark.parametrize("quirk", [0, 1])
def test_columns_match_the_oracle(oracle, columns, rows, slices, quirk):
    from pct_reconstruction_amd import Reconstruction
    P, _ = small_head(n=10, seed=3)
    P, data = small_head(n=20000, seed=91, columns=columns, rows=rows, quirk_voxel_decode=quirk,
                         slice_thickness=P.recon_cyl_height / (slices + 0.5))
    assert P.slices == slices and columns * rows * ((slices + 7) // 8) >= 1 << 18
    ref = oracle.run_pipeline(P, data, stop_after="fbp")
    with Reconstruction(P) as r:
        r.load_histories(data["t"], data["v"], data["u"], data["wepl"], data["angle_deg"])
        r.preprocessing()
        fbp = r.image("fbp").reshape(-1)
    print(f"[fbp {columns}x{rows}x{slices} quirk {quirk}] {np.count_nonzero(fbp != ref['fbp'])} differ", flush=True)
    assert np.array_equal(fbp, ref["fbp"])
