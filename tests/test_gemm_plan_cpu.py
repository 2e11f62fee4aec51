"""The rule that chooses between the stream-K kernel and the library from a table of measured row counts."""

import pytest

from ome_amd import ops


@pytest.mark.parametrize("M,us,lib_us,want", [
    (100, 50, 60, 128),      # one tile, as measured at 128 rows
    (90, 50, 60, None),      # nothing of one tile near enough
    (170, 50, 60, 256),      # two tiles by the 256 rows, not one by the 128 rows
    (256, 50, 51, None),     # as measured: not faster
    (300, 50, 60, 512),      # two tiles of 256 rows by the 512 rows
    (300, 50, 55, None),     # ... which lie further and won by less than a tenth: the 256 rows, times 3 / 2 (82 us)
    (520, 50, 60, None),     # three tiles for the measured two: 75 us for 61
    (520, 50, 100, 512),
    (700, 50, 100, None),
])
def test_row_counts_of_as_many_tiles_speak_first(monkeypatch, M, us, lib_us, want):
    table = [(m, {"bn": 128, "nwg": n, "bm": bm, "us": us, "lib_us": lib_us}) for m, n, bm in ((128, 128, 128), (256, 256, 128), (512, 64, 256))]
    monkeypatch.setattr(ops, "_SK_TABLE", {"1024,512,0": table})
    monkeypatch.setattr(ops, "_SK_MODE", "table")
    plan = ops.gemm_sk_plan(M, 1024, 512, 0)
    assert plan == {None: None, 128: (128, 128, 128), 256: (128, 256, 128), 512: (128, 64, 256)}[want]


def test_every_plan_fits_its_kernel():
    for key in ops._sk_table():
        N, K, epi = map(int, key.split(","))
        for M in range(1, 2600, 7):
            plan = ops.gemm_sk_plan(M, N, K, epi)
            assert plan is None or ops.gemm_sk_ok(M, N, K, *plan)
