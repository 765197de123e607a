"""Chunked admission and ring rewrite (the cache half of a prompt chunk) at the
sizes where the launch's split changes: one to eight 64-position steps per
workgroup, more than 64 heads, chunks that end inside a step, flag rows that
start at any byte and flags other than 0 / 1.  Against the admitted positions
themselves; all copies and integers, bit for bit."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("H,D,W,P,chunks,frac", [
    (1, 64, 64, 16, (64, 64, 65), 0.5),
    (3, 128, 128, 32, (256, 128, 1003), 0.3),
    (8, 128, 1024, 16, (4096, 4096, 1025), 0.2),   # one step per workgroup
    (40, 64, 64, 16, (2048, 4033), 0.2),           # two
    (70, 64, 128, 64, (1024, 8192), 0.1),          # eight
    (2, 64, 64, 16, (640, 640), 0.0),
    (2, 64, 64, 16, (640, 640), 1.0),
    (16, 64, 64, 16, (64, 64, 65), 0.5),           # 16 lanes count a head's flags
    (40, 64, 64, 16, (64, 64, 65), 0.5),           # four
    (130, 64, 64, 16, (64, 64, 65), 0.5),          # one
    (300, 64, 64, 16, (128, 191), 0.3),            # one, two passes over the heads
])
def test_chunks(H, D, W, P, chunks, frac):
    from wgkv import ops
    from wgkv.cache import DualCache
    from wgkv.layers import WGKVConfig
    S, L, layer = sum(chunks), 2, 1
    g = torch.Generator(device=DEV).manual_seed(H * S)
    k, v, pre = (torch.randn(S, H, D, generator=g, device=DEV).to(torch.bfloat16) for _ in range(3))
    flags = (torch.rand(H, S + 3, generator=g, device=DEV) < frac).to(torch.uint8) * \
        torch.randint(1, 256, (H, S + 3), generator=g, device=DEV).to(torch.uint8)
    buf = torch.zeros(1 + flags.numel(), dtype=torch.uint8, device=DEV)
    buf[1:] = flags.flatten()
    mask = buf[1:].view(H, S + 3)[:, :S]  # no row is 16-byte aligned
    adm = mask != 0
    cfg = WGKVConfig(num_hidden_layers=L, num_attention_heads=H, num_key_value_heads=H, head_dim=D, hidden_size=H * D,
                     local_window_size=W, block_size=P, max_tokens_per_head=S + 2 * W,
                     max_total_tokens=L * H * (S + 2 * W), g_defer=True)
    c = DualCache()
    c.initialize(cfg, D, torch.bfloat16, torch.device(DEV))
    print(f"[chunk admit] H{H} D{D} W{W} P{P} {chunks} {frac}", flush=True)
    c0 = 0
    for C in chunks:
        sl = slice(c0, c0 + C)
        step = ops.ChunkStep(c, layer, k[sl], k[sl], v[sl], mask[:, sl], c0, pre_key=pre[sl])
        step.admit()
        cum = torch.cumsum(adm.to(torch.int64), 1)
        for i in range((C + 63) // 64):
            below = (c0 + 64 * i) - W + 1  # admitted positions below the row block's band
            want = cum[:, below - 1] if below > 0 else torch.zeros(H, dtype=torch.int64, device=DEV)
            assert torch.equal(step.column_count[:, i].to(torch.int64), want), (c0, i)
        step.ring()
        c0 += C
    assert int(c.status.item()) == 0
    early, n_loc = S - W, W
    lb = W // P
    used = 0
    for h in range(H):
        idx = adm[h, :early].nonzero().flatten()
        n = idx.numel()
        assert int(c.global_lengths[layer, h]) == n, h
        pages = c.block_table[layer, h, lb:lb + (n + P - 1) // P].long()
        rows = (pages[:, None] * P + torch.arange(P, device=DEV)[None]).flatten()[:n]
        assert torch.equal(c.block_pool_k[rows], k[idx, h]) and torch.equal(c.block_pool_v[rows], v[idx, h]), h
        used += pages.numel()
        ring = torch.arange((layer * H + h) * W, (layer * H + h + 1) * W, device=DEV)
        assert torch.equal(c.block_pool_k[ring], k[S - n_loc:, h]) and torch.equal(c.block_pool_v[ring], v[S - n_loc:, h])
        assert torch.equal(c.local_pre_key[layer, h], pre[S - n_loc:, h])
        assert torch.equal(c.local_is_global[layer, h], adm[h, S - n_loc:])
    ids = torch.cat([c.block_table[layer, h, lb:lb + (int(c.global_lengths[layer, h]) + P - 1) // P] for h in range(H)])
    assert ids.unique().numel() == used and c.next_free_block == L * H * lb + used
