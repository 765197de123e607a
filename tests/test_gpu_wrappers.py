"""The Python wrappers on tensors that are not laid out as the kernels read
them -- strided queries, tables, lengths, outputs and metadata -- and on a
stream that is not the default one: the same kernels on the same values, so
every result must equal the plain layout's bit for bit."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def strided(t, dim):
    """t's values with every second element of a twice as large dim."""
    shape = list(t.shape)
    shape[dim] *= 2
    big = torch.zeros(shape, dtype=t.dtype, device=t.device)
    view = big[tuple(slice(None, None, 2) if d == dim % t.dim() else slice(None) for d in range(t.dim()))]
    view.copy_(t)
    assert view.stride() != t.stride()
    return view


@pytest.mark.parametrize("what", ["q_last", "q_heads", "table", "lens", "out", "stream"])
def test_decode_layouts(what):
    from wgkv import ops, workloads
    w = workloads.decode_ragged(ctx=3000, batch=3, window=256, seed=1)
    args = [w.q, w.k_cache, w.v_cache, w.cache_seqlens, w.block_table.clamp(min=0), w.softmax_scale]
    ref = ops.paged_decode_attn(*args)
    out = None
    if what == "q_last":
        args[0] = strided(w.q, 3)
    elif what == "q_heads":
        args[0] = strided(w.q, 2)
    elif what == "table":
        args[4] = strided(args[4], 2)
    elif what == "lens":
        args[3] = strided(args[3], 1)
    elif what == "out":
        out = strided(torch.zeros_like(ref), 2)
    torch.cuda.synchronize()
    if what == "stream":
        side = torch.cuda.Stream()
        with torch.cuda.stream(side):
            got = ops.paged_decode_attn(*args)
        side.synchronize()
    else:
        got = ops.paged_decode_attn(*args, out=out)
    assert torch.equal(got, ref)


@pytest.mark.parametrize("what", ["metadata", "columns", "out", "heads_first", "mask_uint8"])
def test_prefill_layouts(what):
    import wgkv
    S, H, G, D, W = 1500, 2, 4, 64, 256
    g = torch.Generator(device=DEV).manual_seed(3)
    q, k, v = (torch.randn(1, S, n, D, generator=g, device=DEV).to(torch.bfloat16) for n in (H * G, H, H))
    mask = torch.rand(1, H, S, generator=g, device=DEV) < 0.3
    md = list(wgkv.generate_sparse_indices(mask, W, 1, H, S))
    ref = wgkv.sparse_attn_func(q, k, v, *md)
    out = None
    if what == "metadata":
        md = [strided(md[0], 2), strided(md[1], 3), strided(md[2], 2), md[3]]
    elif what == "columns":
        md[3] = strided(md[3], 3)
    elif what == "out":
        out = torch.zeros(1, H * G, S, D, dtype=torch.bfloat16, device=DEV).transpose(1, 2)
    elif what == "heads_first":
        q, k, v = (t.transpose(1, 2).contiguous().transpose(1, 2) for t in (q, k, v))
    else:
        md = wgkv.generate_sparse_indices(mask.to(torch.uint8) * 7, W, 1, H, S)
    assert torch.equal(wgkv.sparse_attn_func(q, k, v, *md, out=out), ref)


def test_refused_stays_refused():
    import wgkv
    from wgkv import ops, workloads
    w = workloads.decode_ragged(ctx=600, batch=1, window=256, seed=2)
    args = [w.q, w.k_cache, w.v_cache, w.cache_seqlens, w.block_table, w.softmax_scale]
    for i, bad, err in [(0, w.q.cpu(), ValueError), (0, w.q.float(), TypeError), (3, w.cache_seqlens.long(), TypeError),
                        (3, w.cache_seqlens[:, :3], AssertionError), (4, w.block_table[:, :4], AssertionError),
                        (1, w.k_cache[:, :8], AssertionError), (0, w.q[0], AssertionError),
                        (1, torch.cat([w.k_cache, w.k_cache])[::2], ValueError)]:
        with pytest.raises(err):
            ops.paged_decode_attn(*args[:i], bad, *args[i + 1:])
    q = torch.zeros(1, 100, 4, 64, dtype=torch.bfloat16, device=DEV)
    k = torch.zeros(1, 100, 2, 64, dtype=torch.bfloat16, device=DEV)
    md = list(wgkv.generate_sparse_indices(torch.zeros(1, 2, 100, dtype=torch.bool, device=DEV), 64, 1, 2, 100))
    with pytest.raises(AssertionError):
        wgkv.sparse_attn_func(q, k, k, md[0][..., :1], *md[1:])
    with pytest.raises(ValueError):
        wgkv.sparse_attn_func(q.cpu(), k, k, *md)


@pytest.mark.parametrize("call", ["decode", "prefill"])
def test_calls_run_on_the_current_stream(call):
    """The handle is the current stream's, inside and outside a stream context,
    and a call reads what work before it on that stream writes: the queries
    arrive behind a long producer, so a launch on another stream reads zeros."""
    import wgkv
    from wgkv import _lib, ops, workloads
    if call == "decode":
        w = workloads.decode_ragged(ctx=3000, batch=3, window=256, seed=1)
        args = [w.k_cache, w.v_cache, w.cache_seqlens, w.block_table.clamp(min=0), w.softmax_scale]
        fn, q = ops.paged_decode_attn, w.q
    else:
        g = torch.Generator(device=DEV).manual_seed(5)
        q, k, v = (torch.randn(1, 700, n, 64, generator=g, device=DEV).to(torch.bfloat16) for n in (8, 2, 2))
        mask = torch.rand(1, 2, 700, generator=g, device=DEV) < 0.3
        args = [k, v, *wgkv.generate_sparse_indices(mask, 128, 1, 2, 700)]
        fn = wgkv.sparse_attn_func
    ref = fn(q, *args)
    late = torch.zeros_like(q)
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    assert _lib.stream_handle(q.device) == torch.cuda.current_stream(q.device).cuda_stream
    with torch.cuda.stream(side):
        assert _lib.stream_handle(q.device) == side.cuda_stream == torch.cuda.current_stream(q.device).cuda_stream
        torch.cuda._sleep(20_000_000)
        late.copy_(q)
        got = fn(late, *args)
    assert not side.query()  # the call returned before the producer was done
    assert _lib.stream_handle(q.device) == torch.cuda.current_stream(q.device).cuda_stream != side.cuda_stream
    side.synchronize()
    assert torch.equal(got, ref)
