"""``ops.rope_qkv_cache`` at prompt rows: pages whose tokens are all in the call, edges, gaps and padding."""
import pytest
import torch

from ome_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Hq,Hkv,D", [(32, 8, 128), (4, 1, 64), (2, 2, 256)])
@pytest.mark.parametrize("cache", [torch.bfloat16, torch.float8_e4m3fn, torch.float8_e5m2], ids=str)
@pytest.mark.parametrize("T", [511, 512, 700])
def test_prompt_pages(Hq, Hkv, D, cache, T):
    torch.manual_seed(T + D)
    dev, P, pages = "cuda", 16, 64
    run = torch.randperm(pages, device=dev)[:, None] * P + torch.arange(P, device=dev)   # pages in any order
    slots = run.flatten()[5:5 + T].clone()   # begins inside a page
    slots[100:140] = slots[100:140].flip(0)  # no run of a page
    slots[200], slots[300:310] = -1, -1
    slots = slots.int()
    qkv = torch.randn(T, (Hq + 2 * Hkv) * D + 8, device=dev).to(torch.bfloat16)[:, 8:]
    pos = torch.randint(0, 900, (T,), dtype=torch.int32, device=dev)
    ang = torch.rand(900, D // 2, device=dev) * 6
    cs = torch.cat([ang.cos(), ang.sin()], 1).contiguous()
    new = lambda *s: (torch.randn(*s, device=dev) * 0.5).to(cache)  # noqa: E731
    k1, v1 = new(pages, Hkv, P, D), new(pages, Hkv, D, P)
    k2, v2, q1 = k1.clone(), v1.clone(), torch.zeros(T, Hq, D, dtype=torch.bfloat16, device=dev)
    q2, sc = q1.clone(), (1.0, 1.0) if cache == torch.bfloat16 else (0.5, 2.0)
    ops.rope_qkv_cache(qkv, pos, cs, D, q1, k1, v1, slots, Hq, Hkv, D, k_scale=sc[0], v_scale=sc[1])
    for t in range(T):   # the same rows one by one: a token writes its own column
        ops.rope_qkv_cache(qkv[t:t + 1], pos[t:t + 1], cs, D, q2[t:t + 1], k2, v2, slots[t:t + 1], Hq, Hkv, D,
                           k_scale=sc[0], v_scale=sc[1])
    for a, b in ((q1, q2), (k1, k2), (v1, v2)):
        assert torch.equal(a.float(), b.float())
