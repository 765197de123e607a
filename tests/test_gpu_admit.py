"""One-shot admission at the edges of its tiles vs the oracle's state machine:
64-position workgroups, 2048-position count tiles, the ring's boundary, the
number of tiles that moves the counting to its own launch, flag rows that start
at any byte and flags other than 0 / 1.  All outputs are copies and integers:
they must match bit for bit."""
import pytest
import torch

from oracle.dualcache import DualCacheOracle

pytestmark = pytest.mark.gpu
L, LAYER = 2, 1


def run_case(H, S, D, W, P, frac, pad, seed, defer=True):
    from wgkv import ops
    from wgkv.cache import DualCache
    from wgkv.layers import WGKVConfig
    g = torch.Generator().manual_seed(seed)
    key, value, pre = (torch.randn(H, S, D, generator=g).to(torch.bfloat16) for _ in range(3))
    # rows of S + pad flags starting one byte into the buffer: no row is 16-byte aligned
    flags = (torch.rand(H, S + pad, generator=g) < frac).to(torch.uint8) * torch.randint(
        1, 256, (H, S + pad), generator=g, dtype=torch.int32).to(torch.uint8)
    buf = torch.zeros(1 + flags.numel(), dtype=torch.uint8)
    buf[1:] = flags.flatten()
    mask = buf.cuda()[1:].view(H, S + pad)[:, :S]
    per_head = S + 2 * W
    cfg = WGKVConfig(num_hidden_layers=L, num_attention_heads=H, num_key_value_heads=H, head_dim=D, hidden_size=H * D,
                     local_window_size=W, block_size=P, max_tokens_per_head=per_head, max_total_tokens=L * H * per_head,
                     g_defer=defer)
    c = DualCache()
    c.initialize(cfg, D, torch.bfloat16, torch.device("cuda"))
    for t in (c.block_pool_k, c.block_pool_v, c.local_pre_key):
        if t is not None:
            t.zero_()
    print(f"[admit] H{H} S{S} D{D} W{W} P{P} pad{pad}", flush=True)
    ops.prefill_admit(c, LAYER, key.cuda(), value.cuda(), mask, pre_key=pre.cuda() if defer else None)
    o = DualCacheOracle(L, H, D, W, L * H * per_head, per_head, P, g_defer=defer)
    o.prefill(LAYER, key, value, flags[:, :S] != 0, pre)
    assert int(c.status.item()) == 0
    assert c.next_free_block == o.next_free_block
    for name in ("block_table", "global_lengths", "local_is_global", "block_pool_k", "block_pool_v"):
        assert torch.equal(getattr(c, name).cpu(), getattr(o, name)), name
    if defer:
        assert torch.equal(c.local_pre_key.cpu(), o.local_pre_key)


@pytest.mark.parametrize("S", [1, 63, 64, 65, 127, 128, 129, 191, 192, 193, 2047, 2048, 2049, 2175, 2176, 2177, 4225])
@pytest.mark.parametrize("H,D,W,P,pad", [(1, 64, 64, 16, 0), (3, 128, 128, 32, 5)])
def test_tile_edges(H, D, W, P, pad, S):
    run_case(H, S, D, W, P, 0.3, pad, seed=S)


@pytest.mark.parametrize("H,S", [(8, 6144), (8, 6145), (24, 2048), (25, 2048), (70, 300)])
def test_counting_in_the_plan_and_before_it(H, S):
    run_case(H, S, 64, 64, 16, 0.2, 3, seed=H)


@pytest.mark.parametrize("H,S", [(5, 8192), (5, 8193), (70, 130), (130, 65), (200, 2049), (1024, 66)])
def test_threads_per_head_in_the_plan(H, S):
    """Up to four count tiles per head (8192 tokens) and above, and from 5 to
    1024 heads: the plan's threads per head change with the tiles, its passes
    over the heads with their number."""
    run_case(H, S, 16, 16, 16, 0.3, 2, seed=H + S)


@pytest.mark.parametrize("frac", [0.0, 1.0])
def test_none_and_all_admitted(frac):
    run_case(2, 3000, 64, 128, 16, frac, 1, seed=7, defer=False)
