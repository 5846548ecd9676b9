"""Allocations that report no memory (PCT_FAIL_ALLOCATIONS=first,count).  A stage that is refused one says so and can be
run again in the same context, with the same result; what the context keeps only to use it again is given back first
(internal.h: pct_alloc, pct_give_back); the hull counts by image tiles go on by the hash table (k_hull.hip:
carve_by_tiles).
"""
from __future__ import annotations

import numpy as np
import pytest

from cases import small_cylinder, small_head

pytestmark = pytest.mark.gpu


def _load(P, data):
    from pct_reconstruction_amd import Reconstruction
    r = Reconstruction(P)
    r.load_histories(data["t"], data["v"], data["u"], data["wepl"], data["angle_deg"])
    return r


def _allocations(r):
    return r.metrics()["counts"]["device_allocations"]


def _until_it_fits(call):
    """Makes the call again after a refusal for lack of memory; the tries."""
    for tries in range(1, 4):
        try:
            call()
            return tries
        except RuntimeError as e:
            assert "hipMalloc" in str(e)
    raise AssertionError("still no memory")


@pytest.mark.parametrize("method", [0, 1])
def test_a_list_build_without_memory_can_be_run_again(monkeypatch, method):
    P, data = small_cylinder(n=20000, seed=47, drop_block_size=1600, mlp_algorithm=method)
    monkeypatch.setenv("PCT_DROP_TILES", "0")
    with _load(P, data) as r:
        r.preprocessing()
        r.reconstruction_cuts()
        before = _allocations(r)
        r.build_mlp_lists()
        after = _allocations(r)
        r.DROP(2)
        want = r.image("x")
    assert after - before >= 30
    for k in range(before + 1, after + 1):
        print(f"[no memory] list build, allocation {k - before} of {after - before}", flush=True)
        monkeypatch.setenv("PCT_FAIL_ALLOCATIONS", f"{k},1")
        with _load(P, data) as r:
            r.preprocessing()
            r.reconstruction_cuts()
            assert _allocations(r) == before
            assert _until_it_fits(r.build_mlp_lists) == 2
            r.DROP(2)
            assert np.array_equal(r.image("x"), want), k


@pytest.mark.parametrize("refused", range(1, 7))
def test_lists_after_a_refused_larger_build(monkeypatch, tmp_path, refused):
    """The lists of twice the histories are refused an allocation: there are none then, and fewer can be imported."""
    P, data = small_cylinder(n=20000, seed=47, drop_block_size=1600, iterations=2)
    monkeypatch.setenv("PCT_DROP_TILES", "0")

    def twice(r):
        r.load_histories(data["t"], data["v"], data["u"], data["wepl"], data["angle_deg"])
        r.preprocessing()
        r.reconstruction_cuts()

    with _load(P, data) as r:
        want = r.run()
        r.export_preprocessed(tmp_path)
        twice(r)
        k = _allocations(r) + refused
    monkeypatch.setenv("PCT_FAIL_ALLOCATIONS", f"{k},1")
    with _load(P, data) as r:
        r.run()
        r.export_preprocessed(tmp_path)
        twice(r)
        with pytest.raises(RuntimeError, match="hipMalloc"):
            r.build_mlp_lists()
        with pytest.raises(RuntimeError):
            r.DROP(1)
        print(f"[no memory] allocation {refused} of the larger lists refused", flush=True)
        r.import_preprocessed(tmp_path)
        r.DROP(2)
        assert np.array_equal(r.image("x"), want)


def test_the_carve_without_memory_goes_on_by_the_table(monkeypatch):
    P, data = small_head(n=30000, seed=73, columns=70, rows=130, slice_thickness=0.3, sc_on=1)
    monkeypatch.setenv("PCT_CARVE_TILES", "1")
    monkeypatch.setenv("PCT_CARVE_BATCH", "7001")
    kinds = ("sc_hull", "msc_counts", "sm_counts")
    with _load(P, data) as r:
        before = _allocations(r)
        r.import_and_process_data()
        after = _allocations(r)
        assert r.metrics()["carve"]["by_walks"] == 0
        want = [r.image(k) for k in kinds]
    by_table = set()
    for k in range(before + 1, after + 1):
        monkeypatch.setenv("PCT_FAIL_ALLOCATIONS", f"{k},1")
        with _load(P, data) as r:
            _until_it_fits(r.import_and_process_data)
            by_table.add(r.metrics()["carve"]["by_walks"])
            for a, kind in zip(want, kinds):
                assert np.array_equal(a, r.image(kind)), (k, kind)
    print(f"[no memory] {after - before} allocations, histories left to the table {sorted(by_table)}", flush=True)
    assert 30000 in by_table


def test_what_is_kept_is_given_back(monkeypatch):
    """One failed allocation with the carve's scratch in hand: it is freed and the allocation made again."""
    P, data = small_head(n=30000, seed=73, columns=70, rows=130, slice_thickness=0.3)
    monkeypatch.setenv("PCT_CARVE_TILES", "1")
    with _load(P, data) as r:
        r.preprocessing()
        r.reconstruction_cuts()
        before = _allocations(r)
        r.build_mlp_lists()
        r.DROP(2)
        want = r.image("x")
    monkeypatch.setenv("PCT_FAIL_ALLOCATIONS", f"{before + 1},1")
    with _load(P, data) as r:
        r.preprocessing()
        r.reconstruction_cuts()
        assert _allocations(r) == before
        r.build_mlp_lists()
        r.DROP(2)
        assert np.array_equal(r.image("x"), want)
        again = _allocations(r)
        r.import_and_process_data()
        assert _allocations(r) > again  # the scratch is allocated anew
