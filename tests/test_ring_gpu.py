"""Small split-reduction products with every load of a wavefront in flight (ring.hip): each of its tiles, ragged edges, short and
long reductions, residual and views, against fp64."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _close(y, want, size, K):
    """fp32 sums of exact products: a rounding of at most the sum of magnitudes per 32 indices, wavefront and epilogue term."""
    y, want = y.double().cpu().numpy(), want.cpu().numpy()
    bound = size.cpu().numpy() * (K / 32 + 48) * 2.0 ** -24
    assert np.all(np.abs(y - want) <= bound + (np.abs(want) * 2.0 ** -11 + 1e-6)), np.max(np.abs(y - want))


# rows x indices x columns: tiles of 16 x 16 up to 64 x 64, four and eight wavefronts, more pairs than slots and fewer
@pytest.mark.parametrize("M,K,N", [(17, 64, 16), (17, 1024, 4), (31, 4608, 60), (33, 4608, 1000), (100, 256, 2048), (130, 320, 1028),
                                   (400, 128, 1024), (333, 2048, 1000), (500, 1088, 252), (1000, 512, 500), (700, 576, 700),
                                   (2000, 576, 900), (1500, 3584, 260), (3000, 192, 64), (129, 3520, 4100)])
@pytest.mark.parametrize("f16", [False, True])
def test_dense_rows(cuda, oracle, M, K, N, f16):
    from tmq_amd import ops
    print("ring dense", M, K, N, f16, flush=True)
    rng = np.random.default_rng(M + K + N)
    W = rng.integers(-1, 2, size=(N, K)).astype(np.float32)
    nw = ops.NativeWeights(torch.from_numpy(oracle.pack(W).view(np.int32)).to(cuda), N)
    x = torch.from_numpy(rng.standard_normal((M, K)).astype(np.float16)).to(cuda)
    dt = torch.float16 if f16 else torch.float32
    scale, bias = (torch.from_numpy(v.astype(np.float32)).to(cuda) for v in (0.5 + rng.random(N), rng.standard_normal(N)))
    res = torch.from_numpy(rng.standard_normal((M, N)).astype(np.float32)).to(cuda).to(dt)
    xd, wd = x.double().cpu(), torch.from_numpy(W).double()
    plain, size = xd @ wd.t(), xd.abs().sum(1, keepdim=True).expand(M, N)
    y = ops.ternary_linear(x, nw, out_dtype=dt)
    _close(y, plain, size, K)
    full = torch.relu(plain * scale.double().cpu() + bias.double().cpu() + res.double().cpu())
    _close(ops.ternary_linear(x, nw, scale, bias, residual=res, relu=True, out_dtype=dt), full, size * 1.5, K)


@pytest.mark.parametrize("B,C,H,W,N,k,s,p,d", [(1, 64, 56, 56, 64, 3, 1, 1, 1), (1, 512, 7, 7, 512, 3, 1, 1, 1), (4, 64, 56, 56, 128, 1, 2, 0, 1),
                                               (2, 128, 9, 31, 100, 5, 1, 2, 1), (3, 192, 13, 8, 36, 3, 2, 1, 2), (1, 64, 1, 1, 4, 1, 1, 0, 1),
                                               (8, 256, 14, 14, 512, 3, 2, 1, 1), (1, 320, 5, 3, 260, 3, 1, 2, 1)])
@pytest.mark.parametrize("f16", [False, True])
def test_convolutions(cuda, oracle, B, C, H, W, N, k, s, p, d, f16):
    from tmq_amd import ops
    print("ring conv", B, C, H, W, N, k, s, p, d, f16, flush=True)
    gen = torch.Generator().manual_seed(B + C + H + N)
    wt = torch.randint(-1, 2, (N, C, k, k), generator=gen).float()
    nw = ops.NativeWeights(ops.compactify_ternary(wt.to(cuda)), N, conv_kernel=(k, k))
    x = torch.randn(B, C, H, W, generator=gen).half()
    dt = torch.float16 if f16 else torch.float32
    conv = lambda a, b: torch.nn.functional.conv2d(a.double(), b.double(), stride=s, padding=p, dilation=d)
    want, size = conv(x, wt), conv(x.abs(), wt.abs())
    res = torch.randn(want.shape, generator=gen).to(dt)
    xg = x.to(cuda).contiguous(memory_format=torch.channels_last)
    rg = res.to(cuda).contiguous(memory_format=torch.channels_last)
    _close(ops.ternary_conv2d(xg, nw, s, p, d, out_dtype=dt), want, size, C * k * k)
    y = ops.ternary_conv2d(xg, nw, s, p, d, residual=rg, relu=True, out_dtype=dt)
    _close(y, torch.relu(want + res.double()), size, C * k * k)
    # into a strided view of a larger tensor, without the first row of results: the rest untouched
    ho, wo = want.shape[2:]
    big = torch.full((B, N, 2 * ho, 2 * wo), 7.0, device=cuda, dtype=dt).contiguous(memory_format=torch.channels_last)
    first = 1 if ho > 1 else 0
    ops.ternary_conv2d_into(big[:, :, 1:2 * (ho - first):2, 0::2], xg, nw, s, p, d, first=(first, 0))
    _close(big[:, :, 1:2 * (ho - first):2, 0::2], want[:, :, first:], size[:, :, first:], C * k * k)
    assert torch.all(big[:, :, 0::2] == 7.0) and torch.all(big[:, :, :, 1::2] == 7.0)
    assert torch.equal(ops.ternary_conv2d(xg, nw, s, p, d, residual=rg, relu=True, out_dtype=dt), y)


@pytest.mark.parametrize("M,K,N", [(17, 100, 64), (40, 512, 2048), (333, 2000, 1000), (200, 4000, 700), (1000, 256, 1000)])
def test_fp32_row_pairs(cuda, oracle, M, K, N):
    from tmq_amd import ops
    rng = np.random.default_rng(M + K)
    W = rng.integers(-1, 2, size=(N, K)).astype(np.float32)
    nw = ops.NativeWeights(torch.from_numpy(oracle.pack(W).view(np.int32)).to(cuda), N)
    x = rng.standard_normal((M, K)).astype(np.float32) * np.float32(10.0) ** (np.arange(M)[:, None] // 8 % 9 - 4).astype(np.float32)
    want, size = torch.from_numpy(x.astype(np.float64) @ W.T), torch.from_numpy(np.abs(x).astype(np.float64).sum(1, keepdims=True))
    y = ops.ternary_linear(torch.from_numpy(x).to(cuda), nw).double().cpu()
    assert torch.all((y - want).abs() <= size * (2.0 ** -22 + (K / 16 + 64) * 2.0 ** -24))
