#!/usr/bin/env python3
"""Grouped MoE GEMM microbenchmark (gate_up rows compared in token order: the align kernel's
within-expert order is atomic-order dependent) (decode-time shapes): the streamed 64-row tiles vs the 128-row
ones, each in its own process (OME_MOE_TILE); outputs are compared.  Bandwidth = expert weight bytes / time."""
import os
import subprocess
import sys

SHAPES = [  # name, E, H, I, T, k
    ("mixtral-8x7b", 8, 4096, 14336, 256, 2),
    ("qwen3-30b-a3b", 128, 2048, 768, 256, 8),
    ("dsv2-lite", 64, 2048, 1408, 256, 6),
    ("gpt-oss-20b", 32, 2880, 2880, 256, 4),
    ("mixtral-prefill", 8, 4096, 14336, 2048, 2),
    ("qwen3-prefill", 128, 2048, 768, 4096, 8),
    ("mixtral-mid", 8, 4096, 14336, 640, 2),
]


def child():
    import torch

    sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
    from ome_amd import ops

    torch.manual_seed(0)
    dev = "cuda"
    for name, E, H, I, T, k in SHAPES:
        x = torch.randn(T, H, device=dev, dtype=torch.bfloat16)
        w13 = torch.randn(E, 2 * I, H, device=dev, dtype=torch.bfloat16) * 0.02
        w2 = torch.randn(E, H, I, device=dev, dtype=torch.bfloat16) * 0.02
        logits = torch.randn(T, E, device=dev)
        tw, tid = ops.moe_route(logits, k, True)
        n = T * k
        s = ops._Sorted(tid, E, 64)
        inv, tm = s.inv, ops.moe_tile_m(n, E, 2 * I)
        h = torch.randn(n, I, device=dev, dtype=torch.bfloat16)
        gu, y = ops._moe_gemm(x, s, s.ids, k, w13, n, None), ops._moe_gemm(h, s, None, 0, w2, n, None)

        def g1():
            ops._moe_gemm(x, s, s.ids, k, w13, n, None)

        def g2():
            ops._moe_gemm(h, s, None, 0, w2, n, None)

        res = []
        for f, nbytes in ((g1, w13.numel() * 2), (g2, w2.numel() * 2)):
            for _ in range(5):
                f()
            t0, t1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            t0.record()
            for _ in range(30):
                f()
            t1.record()
            torch.cuda.synchronize()
            us = t0.elapsed_time(t1) * 1000 / 30
            res.append(f"{us:8.1f}us {nbytes / us / 1e6:5.2f}TB/s")
        torch.save({"gu": gu.index_select(0, inv.long()).cpu(), "y": y.cpu()}, f"/tmp/moe_{name}_{tm}.pt")
        print(f"tile{tm:<4d}{name:16s} w13 {res[0]} | w2 {res[1]}", flush=True)


def main():
    if len(sys.argv) > 1 and sys.argv[1] == "child":
        return child()
    import torch

    for t in ("64", "128"):
        subprocess.run([sys.executable, __file__, "child"], env={**os.environ, "OME_MOE_TILE": t}, check=True)
    for name, *_ in SHAPES:
        ref, got = (torch.load(f"/tmp/moe_{name}_{v}.pt", weights_only=True) for v in (64, 128))
        err = max((got[t].float() - ref[t].float()).abs().max().item() for t in ("gu", "y"))
        print(f"check {name} 128 vs 64 rows max|diff| = {err:.3e}")
        assert err < 5e-2


if __name__ == "__main__":
    main()
