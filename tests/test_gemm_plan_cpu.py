"""The rules that choose a projection's kernel: between stream-K and the library from a table of measured row counts, and by operands."""

import pytest
import torch

from ome_amd import ops
from ome_amd.models import quant


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


@pytest.mark.parametrize("M,N,K,want", [
    (160, 4096, 4096, (128, 192, 128)),     # 21 us, the library 27: few tiles for the workgroups, so the second row tile costs little
    (520, 4096, 14336, (128, 256, 256)),    # 96 and 112
    (1100, 4096, 14336, None),              # 143 and 154 alone, but whole steps with the library are 2 to 3% shorter
    (300, 6144, 4096, None), (300, 10240, 8192, None), (520, 8192, 28672, None),   # 38 and 29, 94 and 82, 371 and 273
])
def test_plans_by_what_was_measured_between_the_table_s_rows(M, N, K, want):
    assert ops.gemm_sk_plan(M, N, K) == want


class _OnGpu:
    """A tensor that says it is on a GPU."""
    is_cuda = True

    def __init__(self, *shape, dtype=torch.bfloat16, device="cpu"):
        self._t = torch.empty(*shape, dtype=dtype, device=device)

    def __getattr__(self, name):
        return getattr(self._t, name)


@pytest.mark.parametrize("bias,out,M,K,fits", [
    (None, None, 9, 128, True), ((256,), (9, 256), 9, 128, True),
    (None, None, 9, 64, False),        # fewer columns than the weight
    ((1,), None, 9, 128, False), ((128,), None, 9, 128, False), ((9, 256), None, 9, 128, False), ((256, 1), None, 9, 128, False),
    (None, (8, 256), 9, 128, False), (None, (9, 128), 9, 128, False), (None, (9, 512), 9, 128, False),
])
def test_what_is_no_product_is_the_librarys(bias, out, M, K, fits):
    """The kernels take sizes from x and w: a bias or an output of other sizes, and other widths, are refused, resized or broadcast
    by the library as before."""
    x, w = _OnGpu(M, K), _OnGpu(256, 128)
    b, o = (None if s is None else _OnGpu(*s) for s in (bias, out))
    assert ops.gemm_rows_ok(x, w, b, o) == fits
    assert quant._sk_operands_ok(x, w, b, o) == fits


def test_operands_of_other_devices_are_the_librarys():
    x, w, b, o = _OnGpu(9, 128), _OnGpu(256, 128), _OnGpu(256), _OnGpu(9, 256)
    for bad in ((x, w, _OnGpu(256, device="meta"), o), (x, w, b, _OnGpu(9, 256, dtype=torch.float32))):
        assert not ops.gemm_rows_ok(*bad) and not quant._sk_operands_ok(*bad)


# (library or library and activation, this kernel, us)
@pytest.mark.parametrize("N,K,M,epi,want", [
    (27392, 5120, 128, 0, True), (27392, 5120, 160, 0, False), (27392, 5120, 200, 0, True),   # 70 and 79 at 160
    (27392, 5120, 160, 2, True), (28672, 4096, 160, 0, True),
    (49152, 3072, 65, 0, True), (49152, 3072, 80, 0, False), (49152, 3072, 128, 2, True),     # 65 and 70
    (57344, 8192, 128, 0, True), (57344, 8192, 129, 0, False),
    (131072, 1024, 128, 0, True), (128256, 4096, 128, 0, True),
    (256000, 2304, 48, 0, True), (256000, 2304, 64, 0, False),                                # 219 and 235; 245 and 283 at 128
    (53248, 16384, 112, 2, True), (53248, 16384, 128, 2, False),                              # 351 and 396
    (36864, 7168, 9, 0, False),
])
def test_row_kernel_where_it_was_measured_faster(N, K, M, epi, want):
    assert ops.gemm_rows_plan(_OnGpu(M, K, device="meta"), _OnGpu(N, K, device="meta"), epi=epi) == want


@pytest.mark.parametrize("N,K,rows", [
    (4096, 14336, {1, 2, 3, 4, 5, 64, 128, 160, 256}), (4096, 4096, {3, 4, 5, 64, 128, 160}), (5120, 5120, {2, 3, 4, 5, 64, 128, 160, 256}),
    (1536, 8960, {3, 4, 5, 64, 128, 160, 256}), (3584, 3584, {3, 4, 5, 64, 128, 160}), (3072, 3072, {3, 4, 5, 64, 128}), (1024, 4096, {3, 4, 5, 64, 128}),
    (2048, 2048, {4, 5, 64}), (5120, 1024, {3, 4, 5, 64, 128}), (2048, 512, {5, 64, 128}), (8192, 256, set()),
])
def test_pieces_where_they_were_measured_faster(N, K, rows):
    w = _OnGpu(N, K, device="meta")
    assert {M for M in (1, 2, 3, 4, 5, 64, 128, 160, 256) if ops.gemm_rows_parts_plan(_OnGpu(M, K, device="meta"), w)} == rows
