"""Stride-1 convolutions over 128, 256 and 512 channels out of input patches in LDS (patch.hip): shapes inside its lines, with image
and row crossings anywhere in a workgroup's pixels, ragged column groups, dilation and uneven padding, against fp64."""
import pytest
import torch

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


@pytest.mark.parametrize("B,C,H,W,N,k,pad,d", [
    (64, 512, 7, 7, 512, 3, ((1, 1), (1, 1)), 1), (5, 512, 20, 21, 500, 3, ((1, 1), (1, 1)), 1), (3, 512, 30, 31, 440, 3, ((0, 2), (2, 0)), 1),
    (170, 512, 11, 9, 64, 3, ((1, 1), (1, 1)), 1), (64, 256, 14, 14, 256, 3, ((1, 1), (1, 1)), 1), (13, 256, 31, 29, 256, 3, ((1, 1), (1, 1)), 1),
    (20, 256, 24, 22, 248, 3, ((2, 2), (2, 2)), 2), (21, 256, 23, 27, 128, 5, ((2, 2), (2, 2)), 1), (17, 128, 56, 56, 128, 3, ((1, 1), (1, 1)), 1),
    (40, 128, 35, 37, 128, 3, ((0, 0), (0, 0)), 1), (30, 256, 29, 27, 64, 3, ((1, 1), (1, 1)), 1)])
@pytest.mark.parametrize("f16", [False, True])
def test_against_fp64(cuda, oracle, B, C, H, W, N, k, pad, d, f16):
    from tmq_amd import ops
    print("patch conv", B, C, H, W, N, k, pad, d, f16, flush=True)
    gen = torch.Generator(device=cuda).manual_seed(B + C + H + N)
    wt = torch.randint(-1, 2, (N, C, k, k), generator=gen, device=cuda).float()
    nw = ops.NativeWeights(ops.compactify_ternary(wt), N, conv_kernel=(k, k))
    x = torch.randn(B, C, H, W, generator=gen, device=cuda).half().contiguous(memory_format=torch.channels_last)
    dt = torch.float16 if f16 else torch.float32
    want, size = _exact(x, wt, pad, d), _exact(x.abs(), wt.abs(), pad, d)
    # a rounding of at most the sum of magnitudes per 32 indices, slab sum and epilogue term
    bound = size * (C * k * k / 32 + 16) * 2.0 ** -24
    out = bound + want.abs() * (2.0 ** -11 if f16 else 2.0 ** -22)
    y = ops.ternary_conv2d(x, nw, 1, pad, d, out_dtype=dt)
    assert torch.all((y.double() - want).abs() <= out)
    scale, bias = 0.5 + torch.rand(N, generator=gen, device=cuda), torch.randn(N, generator=gen, device=cuda)
    res = torch.randn(want.shape, generator=gen, device=cuda).to(dt).contiguous(memory_format=torch.channels_last)
    full = torch.relu(want * scale.double().view(1, -1, 1, 1) + bias.double().view(1, -1, 1, 1) + res.double())
    y = ops.ternary_conv2d(x, nw, 1, pad, d, scale, bias, residual=res, relu=True, out_dtype=dt)
    assert torch.all((y.double() - full).abs() <= 1.5 * bound + full.abs() * (2.0 ** -11 if f16 else 2.0 ** -21) + 1e-5)
    assert torch.equal(ops.ternary_conv2d(x, nw, 1, pad, d, scale, bias, residual=res, relu=True, out_dtype=dt), y)
