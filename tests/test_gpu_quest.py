"""QUEST on the GPU (through the C ABI): against the reference's own
quest_select_blocks (tests/golden/quest_golden.*: bf16 page scores and fp32)
the token counts, local pages and partial page are exact and the kept full
pages a valid top-k for the reference's scores (equal up to one bf16 step
of the cut, where the reference's topk order is unspecified and an fp32 sum
in another order may round a score to the next bf16 value); against the
oracle, page key bounds after one-shot prefill, chunked prefill and
decode-time promotion are bit-exact, the fp32 selection equals the
oracle's (heads whose cut falls within 1e-5 of a tie are reported, not
compared), and decode attention over the selection matches the fp64
attention over the oracle's selected pages within max-abs 2e-2 / mean-abs
2e-3."""
import types

import pytest
import torch

import scenarios
from oracle import attention, quest
from test_oracle_quest import check_selection_against_golden, quest_gold

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def make_cache(L, H, D, W, mtph):
    from wgkv.cache import DualCache
    from wgkv.layers import WGKVConfig
    cfg = WGKVConfig(num_hidden_layers=L, num_attention_heads=H, num_key_value_heads=H, head_dim=D,
                     hidden_size=H * D, local_window_size=W, block_size=16, max_tokens_per_head=mtph,
                     max_total_tokens=L * H * mtph, use_quest=True, quest_token_budget=256)
    c = DualCache()
    c.initialize(cfg, D, torch.bfloat16, DEV)
    return c


def host_view(c):
    return types.SimpleNamespace(block_table=c.block_table.cpu(), global_lengths=c.global_lengths.cpu(),
                                 block_pool_k=c.block_pool_k.cpu(), block_size=c.block_size,
                                 local_window_size=c.local_window_size)


def assert_bounds_exact(c, layers):
    hv = host_view(c)
    kmin_all, kmax_all = c.quest_block_key_min.cpu(), c.quest_block_key_max.cpu()
    lb = c.local_window_size // c.block_size
    for l in layers:
        for h in range(c.num_kv_heads):
            kmin, kmax = quest.page_bounds(hv, l, h)
            ids = hv.block_table[l, h, lb:lb + kmin.shape[0]].long()
            assert torch.equal(kmin_all[ids].float(), kmin), (l, h)
            assert torch.equal(kmax_all[ids].float(), kmax), (l, h)


def prompt(L, H, S, D, frac, seed):
    g = torch.Generator().manual_seed(seed)
    k = torch.randn(L, H, S, D, generator=g).to(torch.bfloat16)
    v = torch.randn(L, H, S, D, generator=g).to(torch.bfloat16)
    m = torch.rand(L, H, S, generator=g) < frac
    return k.to(DEV), v.to(DEV), m.to(DEV)


@pytest.mark.parametrize("D,frac", [(64, 0.3), (128, 0.6)])
def test_bounds_after_prefill_chunks_and_promotion(D, frac):
    from wgkv import ops
    L, H, W, S = 2, 2, 64, 1000
    print(f"[quest] bounds D{D} admit{frac}", flush=True)
    k, v, m = prompt(L, H, S, D, frac, seed=D)
    c = make_cache(L, H, D, W, S + 200 + W)
    for l in range(L):
        ops.prefill_admit(c, l, k[l], v[l], m[l])
        ops.quest_update_bounds(c, l)
    c.local_length = W
    torch.cuda.synchronize()
    assert_bounds_exact(c, range(L))
    # decode-time promotion: 40 steps, all layers, random flags
    g = torch.Generator().manual_seed(7)
    for step in range(40):
        ops.decode_append(c, 0, migrate=True, write=False)
        for l in range(L):
            kk = torch.randn(H, D, generator=g).to(torch.bfloat16).to(DEV)
            vv = torch.randn(H, D, generator=g).to(torch.bfloat16).to(DEV)
            mm = (torch.rand(H, generator=g) < 0.7).to(DEV)
            ops.decode_append(c, l, kk, vv, g_mask=mm, migrate=False, write=True,
                              cache_seqlens=c.cache_seqlens[l][0])
        c.advance_host_ring()
    torch.cuda.synchronize()
    assert int(c.status.item()) == 0
    assert_bounds_exact(c, range(L))
    # chunked prefill: bounds from the lengths before each chunk
    c2 = make_cache(L, H, D, W, S + W)
    c0 = 0
    for C in (256, 320, 424):
        for l in range(L):
            before = c2.global_lengths[l].clone()
            sl = slice(c0, c0 + C)
            q = torch.randn(C, 2 * H, D, dtype=torch.bfloat16, device=DEV)
            ops.chunk_prefill(c2, l, q, k[l][:, sl].transpose(0, 1), v[l][:, sl].transpose(0, 1), m[l][:, sl], c0)
            ops.quest_update_bounds(c2, l, from_lengths=before)
        c0 += C
    torch.cuda.synchronize()
    assert_bounds_exact(c2, range(L))


@pytest.mark.parametrize("G,D,budget", [(4, 128, 512), (2, 64, 300), (1, 64, 4096), (4, 128, 40)])
def test_selection_matches_oracle(G, D, budget):
    from wgkv import ops
    L, H, W, S = 1, 4, 64, 3000
    print(f"[quest] select G{G} D{D} budget{budget}", flush=True)
    k, v, m = prompt(L, H, S, D, 0.4, seed=G * 100 + D)
    c = make_cache(L, H, D, W, S + W)
    ops.prefill_admit(c, 0, k[0], v[0], m[0])
    ops.quest_update_bounds(c, 0)
    hv = host_view(c)
    g = torch.Generator().manual_seed(budget)
    compared = 0
    for trial in range(5):
        local = [W, 17, 1][trial % 3]
        q = torch.randn(H * G, D, generator=g).to(torch.bfloat16)
        sel_len, sel_bt = ops.quest_select(c, 0, q.to(DEV), local, budget, scores_bf16=False)
        torch.cuda.synchronize()
        o_len, o_blocks = quest.select(hv, 0, q.float(), local, budget, G)
        for h in range(H):
            # skip heads whose cut is a near-tie (fp32 vs fp64 scores)
            n = int(hv.global_lengths[0, h])
            full = n // 16
            kcap = min((max(budget - local, 0) + 15) // 16, (n + 15) // 16) - (1 if n % 16 else 0)
            if 0 < kcap < full:
                kmin, kmax = quest.page_bounds(hv, 0, h)
                s = quest.page_scores(q[h * G:(h + 1) * G].float(), kmin[:full], kmax[:full]).sort(descending=True).values
                if abs(float(s[kcap - 1] - s[kcap])) <= 1e-5 * max(1.0, abs(float(s[kcap]))):
                    print(f"[quest] near tie at the cut, head {h}: not compared", flush=True)
                    continue
            assert int(sel_len[0, h]) == o_len[h], (trial, h)
            got = sel_bt[0, h, :len(o_blocks[h])].cpu().tolist()
            assert got == o_blocks[h], (trial, h)
            compared += 1
    assert compared >= 10


def test_decode_attention_over_selection():
    """Through the layer: use_quest decode steps attend only to the selected
    pages; the output equals fp64 attention over the oracle's selection."""
    from wgkv import layers, ops
    from wgkv.cache import DualCache
    L, H, G, D, W, S, budget = 1, 2, 4, 128, 64, 2000, 320
    print("[quest] layer decode", flush=True)
    cfg = layers.WGKVConfig(num_hidden_layers=L, num_attention_heads=H * G, num_key_value_heads=H, head_dim=D,
                            hidden_size=H * G * D, local_window_size=W, block_size=16,
                            max_total_tokens=L * H * (S + 64 + W), max_tokens_per_head=S + 64 + W,
                            use_quest=True, quest_token_budget=budget)
    s = types.SimpleNamespace(config=cfg, layer_idx=0, head_dim=D, scaling=D ** -0.5, num_key_value_groups=G)
    s.prefill_wrapper = layers.prefill_wrapper
    s.decode_wrapper = layers.decode_wrapper
    s.prefill_kernel = ops.sparse_attn_func
    s.decode_kernel_handle = ops.paged_decode_attn_handle
    s.decode_kernel_executor = lambda f: f()
    g = torch.Generator().manual_seed(11)
    rnd = lambda *sh: torch.randn(*sh, generator=g).to(torch.bfloat16).to(DEV)
    c = DualCache()
    q, k, v = rnd(1, H * G, S, D), rnd(1, H, S, D), rnd(1, H, S, D)
    gm = (torch.rand(1, H, S, generator=g) < 0.3).to(DEV)
    layers.self_attn_forward_patch_inference(s, c, (1, S), q, k, k, v, None, g_mask=gm)
    for step in range(12):
        qi, ki, vi = rnd(1, H * G, 1, D), rnd(1, H, 1, D), rnd(1, H, 1, D)
        mi = (torch.rand(1, H, 1, generator=g) < 0.5).to(DEV)
        local_before = c.local_length
        out = layers.self_attn_forward_patch_inference(s, c, (1, 1), qi, ki, ki, vi, None, g_mask=mi)
        torch.cuda.synchronize()
        # the oracle selection over the cache state this step attended to
        hv = host_view(c)
        local_tokens = min(local_before + 1, W)
        # the layer ranks pages by the reference's bf16 scores (equal scores: lowest page first)
        o_len, o_blocks = quest.select(hv, 0, qi[0, :, 0].float().cpu(), local_tokens, budget, G, scores_bf16=True)
        kc, vc = c.k_cache().cpu().float(), c.v_cache().cpu().float()
        for h in range(H):
            rows_k = kc[o_blocks[h]].reshape(-1, D)[:o_len[h]]
            rows_v = vc[o_blocks[h]].reshape(-1, D)[:o_len[h]]
            for gi in range(G):
                qv = qi[0, h * G + gi, 0].double().cpu()
                w = torch.softmax((rows_k.double() @ qv) * D ** -0.5, dim=0)
                ref = w @ rows_v.double()
                got = out[0, 0, h * G + gi].double().cpu()
                err = (got - ref).abs()
                assert err.max().item() <= 2e-2 and err.mean().item() <= 2e-3, (step, h, gi, err.max().item())


@pytest.mark.parametrize("name", list(scenarios.QUEST_SCENARIOS))
def test_selection_matches_reference_golden(name):
    from wgkv import ops
    z, meta = quest_gold()
    sc = scenarios.QUEST_SCENARIOS[name]
    st = scenarios.quest_state(sc)
    print(f"[quest golden] {name}", flush=True)
    H, D, W, P = sc["H"], sc["D"], sc["W"], 16
    c = types.SimpleNamespace(num_layers=1, num_kv_heads=H, head_dim=D, block_size=P, local_window_size=W,
                              block_table=st["block_table"].to(DEV), global_lengths=st["global_lengths"].to(DEV),
                              quest_block_key_min=st["key_min"].to(torch.bfloat16).to(DEV),
                              quest_block_key_max=st["key_max"].to(torch.bfloat16).to(DEV))
    bf = sc["dtype"] == "bf16"
    for i, (local, budget) in enumerate(sc["steps"]):
        q = st["qs"][i].to(torch.bfloat16).to(DEV)
        sel_len, sel_bt = ops.quest_select(c, 0, q, local, budget, scores_bf16=bf)
        torch.cuda.synchronize()
        rows = []
        budget_blocks = (max(budget - local, 0) + P - 1) // P
        for h, n in enumerate(sc["lengths"]):
            count = (local + P - 1) // P + min(budget_blocks, (n + P - 1) // P)
            rows.append(sel_bt[0, h, :count].cpu().tolist())
        check_selection_against_golden(z, name, i, sc, st, sel_len[0].cpu().tolist(), rows)
    print(f"[quest golden] {name}: {len(sc['steps'])} steps, lengths exact, selections equal up to ties", flush=True)


def check_exact_selection(fulls, G, D, budget, scores_bf16):
    """Heads of `fulls` full pages.  Queries and bounds are small integers, so
    every score is exact in fp32 and ties are many: the selection must be the
    largest scores, equal ones by page order, whole numbers bit for bit."""
    import types
    from wgkv import ops
    W, P = 64, 16
    lens = [f * P + (i % 3) * 5 for i, f in enumerate(fulls)]
    H, lb = len(fulls), W // P
    g = torch.Generator().manual_seed(G * D + budget)
    pages = [(n + P - 1) // P for n in lens]
    total, width = H * lb + sum(pages), lb + max(pages)
    perm = torch.randperm(total, generator=g).to(torch.int32)
    table = torch.full((1, H, width), total - 1, dtype=torch.int32)
    at = 0
    for h, p in enumerate(pages):
        table[0, h, :lb + p] = perm[at:at + lb + p]
        at += lb + p
    lo = torch.randint(-4, 3, (total, D), generator=g).float()
    hi = lo + torch.randint(0, 3, (total, D), generator=g)
    q = torch.randint(-2, 3, (H * G, D), generator=g).float()
    bf = torch.bfloat16
    c = types.SimpleNamespace(num_layers=1, num_kv_heads=H, head_dim=D, block_size=P, local_window_size=W,
                              block_table=table.to(DEV), global_lengths=torch.tensor([lens], dtype=torch.int32).to(DEV),
                              quest_block_key_min=lo.to(bf).to(DEV), quest_block_key_max=hi.to(bf).to(DEV))
    print(f"[quest] exact G{G} D{D} budget{budget} bf16={scores_bf16}", flush=True)
    sel_len, sel_bt = ops.quest_select(c, 0, q.to(bf).to(DEV), W, budget, scores_bf16=scores_bf16)
    cap = (budget - W + P - 1) // P
    for h in range(H):
        full, rem = divmod(lens[h], P)
        have = min(cap, pages[h])
        keep = max(0, min(full, have - (1 if rem else 0)))
        ids = table[0, h, lb:lb + full].long()
        qq = q[h * G:(h + 1) * G, None]
        s = (qq * torch.where(qq >= 0, hi[ids][None], lo[ids][None])).sum(-1)
        s = (s.to(bf).float() if scores_bf16 else s).amax(0)
        order = torch.sort(s, descending=True, stable=True).indices[:keep].sort().values
        want = torch.cat((table[0, h, :lb], table[0, h, lb:][order],
                          table[0, h, lb + full:lb + full + (1 if have > 0 and rem else 0)]))
        assert int(sel_len[0, h]) == W + keep * P + (rem if have > 0 and rem else 0), h
        assert torch.equal(sel_bt[0, h, :want.numel()].cpu(), want), h


@pytest.mark.parametrize("scores_bf16", [False, True])
@pytest.mark.parametrize("G,D", [(1, 128), (3, 64), (4, 128), (5, 8), (8, 256)])
@pytest.mark.parametrize("budget", [64, 64 + 16, 64 + 16 * 40, 64 + 16 * 1500])
def test_selection_exact_over_head_lengths(G, D, budget, scores_bf16):
    """Heads from no page to nearly as many as the selection keeps in LDS
    (12288 pages)."""
    check_exact_selection([0, 1, 15, 16, 17, 63, 64, 65, 1023, 1024, 1025, 2049, 8192, 8193, 12000], G, D, budget,
                          scores_bf16)


@pytest.mark.parametrize("scores_bf16", [False, True])
@pytest.mark.parametrize("G,D", [(1, 128), (4, 64)])
@pytest.mark.parametrize("pages", [1, 2, 3, 64, 159, 160, 161, 255, 256, 257, 6000, 12287, 12288, 12289, 19999])
def test_selection_exact_at_the_edges_of_its_forms(G, D, pages, scores_bf16):
    """Heads ranked page by page (up to 160 or 256 pages), with the keys in LDS
    (up to 12288) and with the scores read again in every step, the budget
    from one page to all but one of each of them."""
    check_exact_selection([2, 3, 65, 159, 160, 161, 255, 256, 257, 258, 12287, 12288, 12289, 20000], G, D,
                          64 + 16 * pages, scores_bf16)


@pytest.mark.parametrize("full,keep", [(f, k) for f in (100, 160, 161, 256, 257, 1000, 12289)
                                       for k in (1, 7, 99, 254) if k < f])
def test_selection_of_distinct_fp32_scores(full, keep):
    """fp32 scores of both signs without ties, where the steps stop early: the
    same pages as the reference's top-k of those scores in 64 bits."""
    import types
    from wgkv import ops
    W, P, D = 64, 16, 8
    lb = W // P
    g = torch.Generator().manual_seed(full + keep)
    # score of page i: q = (1, 2^-8, 0...) on bounds (a_i, b_i) -> distinct for distinct pairs of bf16 integers
    v = torch.randperm(65536, generator=g)[:full] - 32768
    lo = torch.zeros(lb + full, D)
    lo[lb:, 0], lo[lb:, 1] = (v >> 8).float(), (v & 255).float()
    q = torch.zeros(1, D)
    q[0, 0], q[0, 1] = 1.0, 2.0 ** -8
    bf = torch.bfloat16
    table = torch.arange(lb + full, dtype=torch.int32).view(1, 1, -1)
    c = types.SimpleNamespace(num_layers=1, num_kv_heads=1, head_dim=D, block_size=P, local_window_size=W,
                              block_table=table.to(DEV), global_lengths=torch.tensor([[full * P]], dtype=torch.int32).to(DEV),
                              quest_block_key_min=lo.to(bf).to(DEV), quest_block_key_max=lo.to(bf).to(DEV))
    print(f"[quest] distinct full{full} keep{keep}", flush=True)
    sel_len, sel_bt = ops.quest_select(c, 0, q.to(bf).to(DEV), W, W + P * keep, scores_bf16=False)
    want = torch.topk(v.double(), keep).indices.sort().values + lb
    assert int(sel_len[0, 0]) == W + keep * P
    assert torch.equal(sel_bt[0, 0, lb:lb + keep].cpu().long(), want)
