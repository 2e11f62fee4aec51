"""Which kernel, tile and partitions latent attention takes (``ops.MLAWorkspace.tiles``), and that the runtime tells it the
contexts."""
import pytest
import torch

from ome_amd import ops
from ome_amd.models.config import preset
from ome_amd.runtime.model_runner import ModelRunner
from ome_amd.runtime.request import Request, SamplingParams
from ome_amd.runtime.scheduler import ScheduledChunk, StepBatch

W = ops.MLAWorkspace


@pytest.mark.parametrize("T,H,seqs,longest,want", [
    (196, 64, 4, 73, (64, 1)), (400, 16, 4, 100, (32, 1)), (800, 16, 4, 200, (64, 1)), (20, 16, 1, 20, (32, 1)), (8, 16, 1, 308, (0, 64)),
    (100, 64, 1, 3100, (128, 4)), (40, 16, 4, 3010, (64, 11)), (2000, 128, 2, 1000, (128, 1))])
def test_prompts_by_their_longest_context(T, H, seqs, longest, want):
    """... however wide the table is."""
    for width in (-(-longest // 16), 256, 8192):
        rows, decode, parts = ops._latent_tiles(T, H, 576, torch.empty(seqs, width, device="meta"), longest)
        if want[0] == 0:
            assert (rows, decode) == (0, False)
        else:
            assert (rows, decode) == (want[0], False) and want[1] // 2 <= parts <= 2 * want[1], (rows, parts)


@pytest.mark.parametrize("T,H,want", [(1, 128, 0), (2, 128, 0), (3, 128, 32), (12, 128, 64), (32, 128, 128), (64, 128, 0), (4, 64, 0), (6, 64, 32),
                                      (12, 64, 64), (200, 64, 64), (16, 16, 0), (24, 16, 32), (12, 32, 0), (16, 32, 32), (32, 8, 0), (48, 8, 32)])
def test_decode_steps_need_no_context(T, H, want):
    for width in (64, 256, 8192):
        rows, decode, parts = W.tiles(T, H, 576, T, width)
        assert rows == want and decode == (want > 0)
        # a piece's partials: at most 256 pieces of whole tiles, or the other kernels' rows
        assert 256 * rows <= W.ROWS and (rows or T * H * parts <= W.ROWS)


@pytest.mark.parametrize("T,H,pages,want", [(48, 128, 24, 32), (48, 128, 25, 128), (128, 64, 24, 32), (129, 64, 24, 64), (12, 64, 48, 32), (12, 64, 49, 64),
                                            (24, 64, 48, 64), (12, 32, 24, 0), (12, 32, 25, 32), (12, 32, 48, 32), (11, 32, 48, 0)])
def test_decode_steps_over_short_tables(T, H, pages, want):
    """... of which a piece is still one workgroup of the 256."""
    rows, decode, parts = W.tiles(T, H, 576, T, pages)
    assert rows == want and decode == (want > 0)
    assert not rows or (parts == 1 or T * -(-H // rows) <= 256)


def test_many_rows_of_128_heads_fill_the_chip_once():
    for T in (64, 96, 128, 200, 256, 600):
        assert W.tiles(T, 128, 576, T, 256) == (0, False, max(1, 256 // T)) and W.tiles(T, 128, 288, T, 256)[0] == 0


def test_runner_tells_the_longest_context(monkeypatch):
    cfg = preset("tiny-deepseek")
    runner = ModelRunner(cfg, device="cpu", dtype=torch.float32, max_running=4, max_context=512, max_total_tokens=2048, cuda_graph=False)
    seen = []
    attn = ops.mla_attn
    monkeypatch.setattr(ops, "mla_attn", lambda q, *a, max_len=None, **k: (seen.append((q.shape[0], max_len)), attn(q, *a, **k))[1])
    chunks = []
    for i, (past, n) in enumerate([(90, 20), (0, 37), (70, 1), (5, 1)]):
        r = Request([3] * (past + n), SamplingParams(ignore_eos=True))
        r.pages, r.req_slot, r.num_cached = list(range(1 + 8 * i, 9 + 8 * i)), runner.slots.alloc(), past
        runner.slots.set_pages(r.req_slot, 0, r.pages)
        chunks.append(ScheduledChunk(r, past, n, True))
    runner.slots.flush()
    runner.launch(StepBatch("mixed", chunks))
    assert set(seen) == {(57, 110), (2, 71)}
    seen.clear()
    runner.launch(StepBatch("prefill", chunks[:2]))
    assert set(seen) == {(57, 110)}
