"""Stride-1 convolutions over 256 and 512 channels out of input patches in LDS (patch.hip): every instantiation, with image and
row crossings anywhere in a workgroup's pixels, ragged column groups, uneven padding, dilation and windows of several forms,
against fp64. Every shape is one that the patch kernel takes."""
import pytest
import torch

from tests.test_conv_kernels import PATCH, kernel_of

pytestmark = pytest.mark.gpu


def _exact(x, w, pad, d):
    """fp64 convolution as one matrix product per tap, on the GPU."""
    (pt, pb), (pl, pr) = pad
    x = torch.nn.functional.pad(x.double(), (pl, pr, pt, pb))
    ho, wo = x.shape[2] - d * (w.shape[2] - 1), x.shape[3] - d * (w.shape[3] - 1)
    y = 0
    for i in range(w.shape[2]):
        for j in range(w.shape[3]):
            cols = x[:, :, i * d:i * d + ho, j * d:j * d + wo].permute(0, 2, 3, 1).reshape(-1, x.shape[1])
            y = y + cols @ w[:, :, i, j].double().t()
    return y.view(x.shape[0], ho, wo, -1).permute(0, 3, 1, 2)


EVEN = ((1, 1), (1, 1))
# eight slabs; four slabs, two groups of 64 columns and (at most 64 outputs) one; N a multiple of 4 only for fp32 results
SHAPES = [(64, 512, 7, 7, 512, (3, 3), EVEN, 1), (5, 512, 20, 21, 500, (3, 3), EVEN, 1), (170, 512, 11, 9, 64, (3, 3), EVEN, 1),
          (212, 512, 13, 5, 64, (3, 3), ((0, 2), (2, 1)), 1), (62, 512, 26, 11, 64, (3, 3), ((2, 0), (1, 2)), 1),
          (5, 512, 37, 12, 500, (3, 3), ((0, 2), (2, 1)), 1), (20, 512, 38, 6, 256, (4, 4), ((1, 2), (2, 1)), 1),
          (57, 512, 18, 4, 256, (5, 5), ((2, 2), (2, 2)), 1), (191, 512, 31, 4, 64, (9, 1), ((4, 4), (0, 0)), 1),
          (85, 512, 40, 6, 64, (3, 3), ((2, 1), (1, 2)), 2),
          (64, 256, 14, 14, 256, (3, 3), EVEN, 1), (13, 256, 31, 29, 256, (3, 3), EVEN, 1), (20, 256, 24, 22, 248, (3, 3), ((2, 2), (2, 2)), 2),
          (31, 256, 17, 21, 248, (3, 3), ((2, 0), (1, 2)), 1), (102, 256, 34, 5, 248, (3, 3), ((1, 0), (0, 1)), 1),
          (244, 256, 4, 23, 128, (5, 5), ((2, 2), (2, 2)), 1), (105, 256, 25, 10, 192, (3, 3), ((0, 0), (0, 0)), 2),
          (111, 256, 23, 14, 64, (3, 3), EVEN, 1), (102, 256, 24, 14, 64, (3, 3), ((0, 2), (2, 1)), 1),
          (289, 256, 23, 6, 56, (3, 3), ((2, 0), (1, 2)), 1), (285, 256, 21, 6, 64, (4, 4), ((1, 2), (2, 1)), 1),
          (82, 256, 12, 36, 64, (1, 9), ((0, 0), (3, 5)), 1), (147, 256, 17, 15, 60, (3, 3), EVEN, 1)]


@pytest.mark.parametrize("B,C,H,W,N,k,pad,d,f16", [s + (f16,) for s in SHAPES for f16 in (False, True) if s[4] % (8 if f16 else 4) == 0])
def test_against_fp64(cuda, oracle, B, C, H, W, N, k, pad, d, f16):
    from tmq_amd import ops
    print("patch conv", B, C, H, W, N, k, pad, d, f16, flush=True)
    gen = torch.Generator(device=cuda).manual_seed(B + C + H + N)
    assert kernel_of(B, C, H, W, N, k, pad, d, f16=f16) == PATCH
    wt = torch.randint(-1, 2, (N, C, *k), generator=gen, device=cuda).float()
    nw = ops.NativeWeights(ops.compactify_ternary(wt), N, conv_kernel=k)
    x = torch.randn(B, C, H, W, generator=gen, device=cuda).half().contiguous(memory_format=torch.channels_last)
    dt = torch.float16 if f16 else torch.float32
    want, size = _exact(x, wt, pad, d), _exact(x.abs(), wt.abs(), pad, d)
    # a rounding of at most the sum of magnitudes per 32 indices, slab sum and epilogue term
    bound = size * (C * k[0] * k[1] / 32 + 16) * 2.0 ** -24
    out = bound + want.abs() * (2.0 ** -11 if f16 else 2.0 ** -22)
    y = ops.ternary_conv2d(x, nw, 1, pad, d, out_dtype=dt)
    assert torch.all((y.double() - want).abs() <= out)
    scale, bias = 0.5 + torch.rand(N, generator=gen, device=cuda), torch.randn(N, generator=gen, device=cuda)
    res = torch.randn(want.shape, generator=gen, device=cuda).to(dt).contiguous(memory_format=torch.channels_last)
    full = torch.relu(want * scale.double().view(1, -1, 1, 1) + bias.double().view(1, -1, 1, 1) + res.double())
    y = ops.ternary_conv2d(x, nw, 1, pad, d, scale, bias, residual=res, relu=True, out_dtype=dt)
    assert torch.all((y.double() - full).abs() <= 1.5 * bound + full.abs() * (2.0 ** -11 if f16 else 2.0 ** -21) + 1e-5)
    assert torch.equal(ops.ternary_conv2d(x, nw, 1, pad, d, scale, bias, residual=res, relu=True, out_dtype=dt), y)
