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


def test_rounding_of_special_values():
    from wgkv import model_ops
    x = torch.tensor([float("inf"), float("-inf"), 1e-40, 3.3e38, -3.3e38, 0.0, -0.0, 1.0], device="cuda").to(torch.bfloat16)
    a, b = x.repeat_interleave(8)[None], x.repeat(8)[None]
    same(model_ops.silu_mul(a, b), torch.nn.functional.silu(a) * b)
