"""attention's default tiles for launches that 256-row programs do not fill:
lengths at the edges of 64- and 128-row query blocks and 64-key blocks, every
row against float64 (relative norm per row at most 1e-2, as the other attention
tests; the output starts as NaN)."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("B,H,S,D", [(1, 1, 1, 64), (1, 2, 63, 128), (1, 3, 64, 64), (2, 4, 65, 128),
                                     (1, 8, 129, 64), (4, 16, 127, 128), (2, 16, 1000, 64),
                                     (1, 32, 1024, 128), (5, 8, 300, 128), (4, 32, 520, 64)])
def test_small_launches(B, H, S, D, causal):
    from newt_amd import workloads as W
    g = torch.Generator(device="cuda").manual_seed(S)
    q, k, v = (torch.randn(B, H, S, D, generator=g, device="cuda").bfloat16() for _ in range(3))
    o = torch.full_like(q, float("nan"))
    print(f"attention tile {W.attention_tile(S, B * H, D, causal)} for {B}x{H}x{S}x{D}", flush=True)
    W.attention(q, k, v, causal=causal, out=o)
    for b in range(B):
        for h in range(H):
            s = q[b, h].double() @ k[b, h].double().t().contiguous() * D ** -0.5
            if causal:
                s.masked_fill_(torch.ones(S, S, dtype=torch.bool, device="cuda").triu(1),
                               float("-inf"))
            ref = torch.softmax(s, -1) @ v[b, h].double()
            err = (o[b, h].double() - ref).norm(dim=1) / ref.norm(dim=1)
            assert float(err.max()) <= 1e-2, (b, h)


@pytest.mark.parametrize("S", [128, 300])
def test_wide_heads_on_four_waves(S):
    """256-wide heads on 128 rows, which large causal launches of them take."""
    from newt_amd import workloads as W
    g = torch.Generator(device="cuda").manual_seed(S)
    q, k, v = (torch.randn(1, 2, S, 256, generator=g, device="cuda").bfloat16() for _ in range(3))
    o = W.attention(q, k, v, causal=True, BLOCK_M=128, num_warps=4)
    for h in range(2):
        s = q[0, h].double() @ k[0, h].double().t().contiguous() / 16
        s.masked_fill_(torch.ones(S, S, dtype=torch.bool, device="cuda").triu(1), float("-inf"))
        ref = torch.softmax(s, -1) @ v[0, h].double()
        err = (o[0, h].double() - ref).norm(dim=1) / ref.norm(dim=1)
        assert float(err.max()) <= 1e-2, h
