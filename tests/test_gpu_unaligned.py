"""Vector accesses at an element's own alignment and under masks that a run of
elements straddles, on copies (bit-exact, guard elements around the output
unchanged) and on the row kernels against float64 at their usual tolerances."""

import pytest
import torch

import newt
import newt.language as nl

pytestmark = pytest.mark.gpu


@newt.jit
def copy_rows_k(x_ptr, o_ptr, N, first, stride, BLOCK: nl.constexpr):
    row = nl.program_id(0)
    cols = nl.arange(0, BLOCK)
    mask = (cols < N) & (cols >= first)
    v = nl.load(x_ptr + row * stride + cols, mask=mask, other=0)
    nl.store(o_ptr + row * stride + cols, v, mask=mask)


@newt.jit
def copy_prefix_k(x_ptr, o_ptr, N, stride, BLOCK: nl.constexpr):
    row = nl.program_id(0)
    cols = nl.arange(0, BLOCK)
    mask = cols < N
    v = nl.load(x_ptr + row * stride + cols, mask=mask, other=7)
    nl.store(o_ptr + row * stride + cols, v, mask=mask)


@pytest.mark.parametrize("dtype", [torch.int8, torch.float16, torch.float32, torch.int64])
@pytest.mark.parametrize("offset", [0, 1, 3])
@pytest.mark.parametrize("N,first,stride", [(1, 0, 1), (255, 0, 257), (256, 0, 256), (250, 3, 255),
                                            (254, 0, 260), (248, 8, 256), (5, 5, 9),
                                            (240, 0, 250)])
def test_masked_copies_are_exact(dtype, offset, N, first, stride):
    rows, pad = 3, 300
    g = torch.Generator(device="cuda").manual_seed(2)
    src = torch.randint(-100, 100, (rows * stride + pad + offset,), generator=g,
                        device="cuda").to(dtype)
    for prefix in (False, True):
        if prefix and first:
            continue
        dst = torch.full_like(src, 101)
        x, o = src[offset:], dst[offset:]
        if prefix:
            copy_prefix_k[(rows,)](x, o, N, stride, BLOCK=256)
        else:
            copy_rows_k[(rows,)](x, o, N, first, stride, BLOCK=256)
        want = torch.full_like(src, 101)
        for r in range(rows):
            a = offset + r * stride
            want[a + first:a + N] = src[a + first:a + N]
        assert torch.equal(dst, want), prefix


@pytest.mark.parametrize("M,N", [(5, 781), (3, 1001), (2, 1002), (4, 1000), (3, 4), (2, 8191)])
@pytest.mark.parametrize("offset", [0, 1])
def test_row_kernels_on_odd_rows(M, N, offset):
    from newt_amd import workloads as W
    g = torch.Generator(device="cuda").manual_seed(3)
    x = torch.randn(M * N + offset, generator=g, device="cuda")[offset:].view(M, N) * 4
    if offset:
        base = torch.empty(M * N + 1, device="cuda")
        base[1:].copy_(x.reshape(-1))
        x = base[1:].view(M, N)
    y = W.softmax(x)
    ref = torch.softmax(x.double(), -1)
    assert bool(((y.double() - ref).abs() <= 1e-5 * ref + 1e-30).all())
    h = x.half()
    w = torch.randn(N, generator=g, device="cuda").half()
    b = torch.randn(N, generator=g, device="cuda").half()
    out, mean, rstd = W.layernorm(h, w, b)
    ref = torch.nn.functional.layer_norm(h.double(), (N,), w.double(), b.double(), 1e-5)
    # half an fp16 ulp of the result (2^-11 relative, 2^-25 absolute) and the
    # fp32 error of its terms
    bound = 2.0 ** -11 * ref.abs() + 2.0 ** -24 + 1e-5 * (ref - b.double()).abs() + 1e-6 * b.abs()
    assert bool(((out.double() - ref).abs() <= bound).all())


@newt.jit
def padded_rows_k(x_ptr, o_ptr, N, stride, NEGATIVE: nl.constexpr, OTHER: nl.constexpr,
                  BLOCK: nl.constexpr):
    row = nl.program_id(0)
    cols = nl.arange(0, BLOCK)
    if NEGATIVE:
        v = nl.load(x_ptr + row * stride + cols, mask=cols < N, other=-0.0)
    else:
        v = nl.load(x_ptr + row * stride + cols, mask=cols < N, other=OTHER)
    nl.store(o_ptr + row * BLOCK + cols, v)


@pytest.mark.parametrize("other", [0.0, -0.0, 2.5, float("-inf")])
@pytest.mark.parametrize("N", [16, 240, 250, 256])
def test_fill_value_keeps_its_bits(N, other):
    g = torch.Generator(device="cuda").manual_seed(4)
    x = torch.randn(3, 272, generator=g, device="cuda")
    o = torch.full((3, 256), float("nan"), device="cuda")
    padded_rows_k[(3,)](x, o, N, 272, NEGATIVE=str(other) == "-0.0", OTHER=other, BLOCK=256,
                        num_warps=1)
    want = torch.full((3, 256), other, device="cuda")
    want[:, :N] = x[:, :N]
    assert torch.equal(o.view(torch.int32), want.view(torch.int32))
