"""The packed gate's two tile sizes (32 and 64 tokens per workgroup): a token's
score does not depend on how many tokens the call holds, so a short call's
scores and flags -- at the edges of both tiles and on both sides of the grid
size that changes them -- must equal the same tokens' in a long call bit for
bit."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("param", ["bf16", "fp32"])
@pytest.mark.parametrize("H,D,inputs,expand,fast", [(8, 128, ["pre_k", "post_k"], 4.0, False),
                                                    (3, 64, ["pre_k", "post_k", "v"], 1.5, True),
                                                    (8, 128, ["post_k"], 1.5, True)])
def test_short_calls_equal_the_long_one(H, D, inputs, expand, fast, param):
    from wgkv.gate import GatingPredictor
    torch.manual_seed(D)
    gate = GatingPredictor(D, H, inputs, "gelu", expand, 1e-3, True, fast).to(
        "cuda", torch.bfloat16 if param == "bf16" else torch.float32)
    S = 64 * (256 // H) + 700  # more 64-token workgroups than a card has CUs
    g = torch.Generator(device="cuda").manual_seed(H)
    x = [torch.randn(1, H, S, D, generator=g, device="cuda").to(torch.bfloat16) for _ in range(3)]
    scores, mask = gate.scores_and_mask(*x, 0.5)
    for n in (5, 31, 32, 33, 63, 64, 65, 1000, 64 * (256 // H) - 1, 64 * (256 // H), 64 * (256 // H) + 1):
        print(f"[gate tiles] H{H} D{D} {param} {n}", flush=True)
        s, m = gate.scores_and_mask(*(t[:, :, S - n:] for t in x), 0.5)
        assert torch.equal(s, scores[:, :, S - n:]) and torch.equal(m, mask[:, :, S - n:]), n
