"""softmax and layernorm over rows short enough for several to a program: row
counts around a program's, widths at the edges of the rule, against float64 at
the tolerances of the other row-kernel tests."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def rnd(*shape, dtype, seed, scale=1.0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return (torch.randn(*shape, generator=g, device="cuda") * scale).to(dtype)


@pytest.mark.parametrize("N", [1, 3, 4, 7, 33, 64, 65, 128, 129, 255, 256, 257])
@pytest.mark.parametrize("M", [1, 15, 17, 1000])
def test_softmax(M, N):
    from newt_amd import workloads as W
    x = rnd(M, N, dtype=torch.float32, seed=M + N, scale=4.0)
    out = torch.full((M + 1, N), float("nan"), device="cuda")
    W.softmax(x, out=out[:M])
    ref = torch.softmax(x.double(), -1)
    assert bool(((out[:M].double() - ref).abs() <= 1e-5 * ref + 1e-30).all())
    assert bool(out[M].isnan().all())


def test_softmax_special_rows():
    """Rows that are constant, hold -inf, or only -inf (0 / 0, as a row per
    program gives)."""
    from newt_amd import workloads as W
    x = rnd(40, 100, dtype=torch.float32, seed=1)
    x[3] = 7.0
    x[5, ::2] = float("-inf")
    x[6] = float("-inf")
    x[7, 9] = float("nan")
    got, want = W.softmax(x), W.softmax(x, num_warps=2)
    assert torch.equal(got.isnan(), want.isnan())
    torch.testing.assert_close(got, want, rtol=1e-6, atol=0, equal_nan=True)


@pytest.mark.parametrize("dtype,N", [(torch.float32, 5), (torch.float32, 256), (torch.float16, 8),
                                     (torch.float16, 511), (torch.float16, 512),
                                     (torch.bfloat16, 65), (torch.bfloat16, 513)])
@pytest.mark.parametrize("M", [1, 7, 129])
def test_layernorm(M, N, dtype):
    from newt_amd import workloads as W
    x, w, b = (rnd(*s, dtype=dtype, seed=i) for i, s in enumerate(((M, N), (N,), (N,))))
    out, mean, rstd = W.layernorm(x, w, b)
    X = x.double()
    m = X.mean(1)
    r = ((X - m[:, None]).square().mean(1) + 1e-5).rsqrt()
    assert bool(((mean.double() - m).abs() <= 1e-5 * m.abs() + 1e-7 * X.abs().mean(1)).all())
    assert bool(((rstd.double() - r).abs() <= 1e-5 * r).all())
    t = (X - m[:, None]) * r[:, None] * w.double()
    ref = t + b.double()
    # half an ulp of the output type, and the fp32 error of the two terms
    half = {torch.float32: 2.0 ** -24, torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}[dtype]
    bound = half * ref.abs() + 2.0 ** -24 + 1e-5 * t.abs() + 1e-6 * b.double().abs()
    assert bool(((out.double() - ref).abs() <= bound).all())
