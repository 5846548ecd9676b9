"""An import of preprocessed data that stops half-way, its path file missing, leaves no lists to run on: the arrays of
an earlier run are overwritten by then (pct_import_preprocessed; init_import_preprocessed_data, V.cu:6775).  The loaded
histories can still be reconstructed."""
from __future__ import annotations

import numpy as np
import pytest

from cases import small_cylinder

pytestmark = pytest.mark.gpu


def test_an_import_that_stops_leaves_no_lists(tmp_path):
    from pct_reconstruction_amd import Reconstruction
    P, data = small_cylinder(n=20000, seed=9)
    with Reconstruction(P) as r:
        r.load_histories(data["t"], data["v"], data["u"], data["wepl"], data["angle_deg"])
        want = r.run()
        r.export_preprocessed(tmp_path)
        (tmp_path / "MLP.bin").rename(tmp_path / "MLP.kept")
        with pytest.raises(RuntimeError):
            r.import_preprocessed(tmp_path)
        with pytest.raises(RuntimeError):
            r.DROP(1)
        assert np.array_equal(r.run(), want)
        (tmp_path / "MLP.kept").rename(tmp_path / "MLP.bin")
        r.import_preprocessed(tmp_path)
        r.DROP(P.iterations)
        assert np.array_equal(r.image("x"), want)
