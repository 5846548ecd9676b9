"""A DROP plan over image tiles whose allocations report no memory (PCT_FAIL_ALLOCATIONS=first,count) becomes one of
sorted lists (k_drop2.hip: pct_drop_prepare), with the same image: lists that change the tile at every step take
more memory over tiles than sorted.
"""
from __future__ import annotations

import numpy as np
import pytest

from cases import small_cylinder
from test_no_memory import _allocations, _load, _until_it_fits

pytestmark = pytest.mark.gpu


def test_a_plan_over_tiles_without_memory_becomes_sorted_lists(monkeypatch):
    P, data = small_cylinder(n=30000, seed=47, drop_block_size=1600)
    monkeypatch.setenv("PCT_DROP_TILES", "1")
    with _load(P, data) as r:
        r.preprocessing()
        r.reconstruction_cuts()
        before = _allocations(r)
        r.build_mlp_lists()
        after = _allocations(r)
        assert r.metrics()["drop_plan"]["tiles"]
        r.DROP(2)
        want = r.image("x")
    fell_back = refused = 0
    for k in range(before + 1, after + 1):
        monkeypatch.setenv("PCT_FAIL_ALLOCATIONS", f"{k},2")  # and once more after what is kept was given back
        with _load(P, data) as r:
            r.preprocessing()
            r.reconstruction_cuts()
            assert _allocations(r) == before
            tries = _until_it_fits(r.build_mlp_lists)
            refused += tries > 1
            fell_back += not r.metrics()["drop_plan"]["tiles"]
            r.DROP(2)
            assert np.array_equal(r.image("x"), want), k
    print(f"[no memory] {after - before} allocations: {fell_back} plans by sorted lists, {refused} refused", flush=True)
    assert fell_back >= 15
