"""The rotary launch's split of tokens over workgroups (several tokens per
workgroup, one, or several workgroups per token) against the torch composition
in the same bf16 rounding, bit for bit, with infinities, NaN and the smallest
and largest bf16 magnitudes among the inputs."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def same(a, b):
    nan = torch.isnan(b)
    assert torch.equal(torch.isnan(a), nan)
    assert torch.equal(a[~nan], b[~nan])


@pytest.mark.parametrize("B,S", [(1, 1), (1, 5), (2, 33), (1, 1000)])
@pytest.mark.parametrize("Hq,Hkv,D", [(1, 1, 16), (2, 1, 32), (8, 2, 64), (3, 3, 48), (28, 4, 128), (48, 8, 128),
                                      (56, 8, 128), (64, 8, 128), (64, 8, 256)])
def test_split_matches_torch(B, S, Hq, Hkv, D):
    from wgkv import model_ops
    from wgkv.attention import apply_rotary_pos_emb
    g = torch.Generator(device="cuda").manual_seed(Hq * D + S)
    buf = torch.randn(B, S, Hq + 2 * Hkv, D, generator=g, device="cuda").to(torch.bfloat16)
    special = torch.tensor([float("inf"), float("-inf"), float("nan"), 1e-40, 3.3e38, 0.0, -0.0],
                           device="cuda").to(torch.bfloat16)
    where = torch.randint(0, buf.numel(), (7 * 4,), generator=g, device="cuda")
    buf.view(-1)[where] = special.repeat(4)
    q, k, v = (t.transpose(1, 2) for t in (buf[:, :, :Hq], buf[:, :, Hq:Hq + Hkv], buf[:, :, Hq + Hkv:]))
    ang = torch.rand(B, S, D, generator=g, device="cuda") * 6.28
    cos, sin = ang.cos().to(torch.bfloat16), ang.sin().to(torch.bfloat16)
    print(f"[rope split] B{B} S{S} Hq{Hq} Hkv{Hkv} D{D}", flush=True)
    qo, ko, vo = model_ops.rope_qkv(q, k, v, cos, sin)
    qr, kr = apply_rotary_pos_emb(q, k, cos, sin)
    same(qo, qr)
    same(ko, kr)
    same(vo, v)


@pytest.mark.parametrize("S", [1, 37])
@pytest.mark.parametrize("Hq,Hkv,D", [(1, 1, 48), (5, 2, 80), (8, 2, 96), (3, 3, 112), (2, 1, 176), (48, 8, 240),
                                      (1, 1, 16), (8, 2, 32), (64, 8, 128), (64, 8, 256)])
def test_head_norms_over_head_dims(Hq, Hkv, D, S):
    """The per-head norm for every multiple of 16 up to 256, where the threads
    of a head are a power of two and where they are not, one or several
    workgroups per token.  The normalised k is within a bf16 step of the torch
    norm (its sum of squares is summed in another order: relative 1.5 * 2^-7
    with the weight's rounding) and rotates to exactly the rotated k; the
    rotated q is within 2^-5 of its operands' magnitudes."""
    from wgkv import model_ops
    from wgkv.attention import apply_rotary_pos_emb
    g = torch.Generator(device="cuda").manual_seed(Hq * D + S)
    # heads of different magnitudes: a sum over another head's elements shows
    buf = torch.randn(1, S, Hq + 2 * Hkv, D, generator=g, device="cuda")
    buf = (buf * torch.exp(2 * torch.randn(1, S, Hq + 2 * Hkv, 1, generator=g, device="cuda"))).to(torch.bfloat16)
    q, k, v = (t.transpose(1, 2) for t in (buf[:, :, :Hq], buf[:, :, Hq:Hq + Hkv], buf[:, :, Hq + Hkv:]))
    ang = torch.rand(1, S, D, generator=g, device="cuda") * 6.28
    cos, sin = ang.cos().to(torch.bfloat16), ang.sin().to(torch.bfloat16)
    qw, kw = ((1 + 0.1 * torch.randn(D, generator=g, device="cuda")).to(torch.bfloat16) for _ in range(2))
    print(f"[rope split] norms Hq{Hq} Hkv{Hkv} D{D} S{S}", flush=True)

    def norm(x, w):
        xf = x.float()
        return w * (xf * torch.rsqrt(xf.pow(2).mean(-1, keepdim=True) + 1e-6)).to(torch.bfloat16)

    qo, ko, vo, kp = model_ops.rope_qkv(q, k, v, cos, sin, qw, kw, 1e-6)
    qn, kn = norm(q, qw), norm(k, kw)
    assert ((kp.float() - kn.float()).abs() <= 1.5 * 2 ** -7 * kn.float().abs()).all()
    qr, kr = apply_rotary_pos_emb(qn, kp, cos, sin)
    same(ko, kr)
    same(vo, v)
    mag = qn.float().abs()
    mag = mag + torch.cat((mag[..., D // 2:], mag[..., :D // 2]), -1)
    assert ((qo.float() - qr.float()).abs() <= 2 ** -5 * mag).all()


def test_more_threads_than_one_launch_holds():
    """129 threads of each token in workgroups of 192: more than 2^32 threads
    for 25 million tokens, so the call takes several launches.  Every token
    reads the same rows (strides of 0) and writes its own k row."""
    from wgkv import _lib
    S, Hq, Hkv, D = 25_000_000, 41, 1, 48
    g = torch.Generator(device="cuda").manual_seed(5)
    x = torch.randn(Hq + 2 * Hkv, D, generator=g, device="cuda").to(torch.bfloat16)
    cos, sin = (torch.randn(D, generator=g, device="cuda").to(torch.bfloat16) for _ in range(2))
    out = torch.zeros(Hq + 2 * Hkv, D, dtype=torch.bfloat16, device="cuda")
    ko = torch.full((S, D), float("nan"), dtype=torch.bfloat16, device="cuda")
    q, k, v, qo, vo = x[:Hq], x[Hq:Hq + 1], x[Hq + 1:], out[:Hq], out[Hq + 1:]
    row = (0, 0, D)
    print("[rope split] 25M tokens", flush=True)
    st = _lib.lib().wgkv_rope_qkv(
        q.data_ptr(), *row, k.data_ptr(), *row, v.data_ptr(), *row, cos.data_ptr(), sin.data_ptr(), 0, 0,
        qo.data_ptr(), *row, ko.data_ptr(), 0, D, D, vo.data_ptr(), *row, 1, S, Hq, Hkv, D,
        _lib.stream_handle(x.device))
    torch.cuda.synchronize()
    assert st == 0

    def rot(t):
        return t * cos + torch.cat((-t[..., D // 2:], t[..., :D // 2]), -1) * sin

    assert torch.equal(qo, rot(q)) and torch.equal(vo, v)
    assert torch.equal(ko[:1], rot(k)) and bool((ko == ko[:1]).all())


def test_rounding_of_special_values():
    from wgkv import model_ops
    x = torch.tensor([float("inf"), float("-inf"), 1e-40, 3.3e38, -3.3e38, 0.0, -0.0, 1.0], device="cuda").to(torch.bfloat16)
    a, b = x.repeat_interleave(8)[None], x.repeat(8)[None]
    same(model_ops.silu_mul(a, b), torch.nn.functional.silu(a) * b)
