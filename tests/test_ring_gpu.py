"""Small split-reduction products with every load of a wavefront in flight (ring.hip): each of its tiles as rows, fp32 row pairs
and convolutions, ragged edges, short and long reductions, residual and views, and what stays with mid.hip or the tile kernels
around them, against fp64. Every shape says which kernel and tile takes it."""
import numpy as np
import pytest
import torch

from tests.test_conv_kernels import kernel_of

pytestmark = pytest.mark.gpu
MID, TILES = 1 - 16, -16   # tmq_ternary_rows_kernel's answers less TMQ_KERNEL_RING


def _close(y, want, size, K):
    """fp32 sums of exact products: a rounding of at most the sum of magnitudes per 32 indices, wavefront and epilogue term, and
    the result's own rounding."""
    ulp = 2.0 ** -11 if y.dtype == torch.float16 else 2.0 ** -22
    y, want = y.double().cpu().numpy(), want.cpu().numpy()
    bound = size.cpu().numpy() * (K / 32 + 48) * 2.0 ** -24
    assert np.all(np.abs(y - want) <= bound + (np.abs(want) * ulp + 1e-6)), np.max(np.abs(y - want))


# rows x indices x columns: tiles of 16 x 16 up to 64 x 64, four and eight wavefronts, more pairs than slots and fewer
@pytest.mark.parametrize("M,K,N,tile", [(17, 64, 16, 0), (22, 256, 12, 0), (17, 1024, 4, 1), (31, 4608, 60, 1), (33, 4608, 1000, 1),
                                        (35, 64, 1448, 2), (607, 128, 132, 2), (40, 704, 1384, 3), (500, 1088, 252, 3),
                                        (100, 256, 2048, 4), (355, 128, 472, 4), (3000, 192, 64, 4), (130, 320, 1028, 5),
                                        (3979, 640, 36, 5), (34, 192, 4564, 6), (78, 704, 3108, 6), (295, 960, 1252, 7),
                                        (33, 896, 5972, 7), (1000, 512, 500, 8), (700, 576, 700, 8), (126, 576, 3372, 8),
                                        (2000, 576, 900, 9), (293, 896, 3576, 9), (129, 3520, 4100, 10), (2474, 1984, 216, 10),
                                        (333, 2048, 1000, MID), (1500, 3584, 260, MID), (97, 4096, 1028, MID), (621, 704, 1540, MID),
                                        (37, 2304, 2000, MID), (400, 128, 1024, TILES)])
@pytest.mark.parametrize("f16", [False, True])
def test_dense_rows(cuda, oracle, M, K, N, tile, f16):
    from tmq_amd import _capi, ops
    assert _capi.load().tmq_ternary_rows_kernel(_capi.F16, M, K, N) == 16 + tile
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


@pytest.mark.parametrize("B,C,H,W,N,k,s,p,d,tile", [
    (1, 64, 1, 1, 4, 1, 1, 0, 1, 0), (11, 192, 5, 3, 4, 1, 2, 0, 1, 0), (1, 512, 7, 7, 512, 3, 1, 1, 1, 1), (2, 128, 9, 31, 100, 5, 1, 2, 1, 1),
    (3, 192, 13, 8, 36, 3, 2, 1, 2, 1), (1, 320, 5, 3, 260, 3, 1, 2, 1, 1), (7, 128, 1, 37, 228, 1, 2, 1, 2, 2), (10, 128, 13, 23, 76, 1, 2, 0, 1, 2),
    (3, 128, 28, 23, 40, 2, 1, 0, 2, 3), (4, 128, 14, 38, 28, 2, 1, 1, 1, 3), (8, 192, 35, 9, 72, 1, 1, 0, 2, 4), (6, 64, 36, 28, 24, 2, 1, 0, 1, 4),
    (1, 64, 56, 56, 64, 3, 1, 1, 1, 5), (8, 256, 14, 14, 512, 3, 2, 1, 1, 5), (1, 128, 37, 27, 172, 2, 1, 0, 2, 5),
    (3, 128, 22, 40, 268, 1, 2, 0, 1, 6), (2, 128, 29, 12, 204, 1, 1, 1, 1, 6), (3, 128, 21, 7, 664, 3, 1, 1, 1, 7), (9, 192, 13, 38, 44, 3, 1, 1, 1, 7),
    (5, 64, 31, 13, 232, 3, 1, 1, 2, 8), (3, 512, 8, 41, 420, 1, 1, 0, 2, 8), (5, 64, 15, 38, 476, 3, 1, 0, 1, 9), (13, 64, 27, 53, 36, 3, 1, 1, 2, 9),
    (9, 192, 11, 19, 324, 3, 1, 1, 1, 10), (10, 192, 57, 3, 356, 3, 1, 1, 1, 10), (3, 512, 11, 31, 120, 3, 1, 1, 1, MID), (3, 512, 27, 18, 332, 2, 1, 0, 1, MID), (4, 64, 56, 56, 128, 1, 2, 0, 1, TILES)])
@pytest.mark.parametrize("f16", [False, True])
def test_convolutions(cuda, oracle, B, C, H, W, N, k, s, p, d, tile, f16):
    from tmq_amd import ops
    assert kernel_of(B, C, H, W, N, (k, k), p, d, s, f16) == 16 + tile
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


@pytest.mark.parametrize("M,K,N,tile", [(17, 100, 64, 0), (55, 192, 4, 0), (23, 590, 36, 1), (26, 16, 1032, 2), (163, 128, 236, 2),
                                        (276, 664, 124, 3), (63, 65, 1112, 4), (989, 100, 104, 4), (40, 512, 2048, 5), (423, 655, 168, 5),
                                        (69, 408, 3688, 6), (200, 4000, 700, 7), (142, 1122, 1052, 7), (318, 576, 692, 8), (950, 495, 984, 9),
                                        (333, 2000, 1000, 10), (210, 1984, 1244, 10), (75, 4096, 4096, MID), (1000, 256, 1000, TILES)])
def test_fp32_row_pairs(cuda, oracle, M, K, N, tile):
    from tmq_amd import _capi, ops
    assert _capi.load().tmq_ternary_rows_kernel(_capi.F32, M, K, N) == 16 + tile
    rng = np.random.default_rng(M + K)
    W = rng.integers(-1, 2, size=(N, K)).astype(np.float32)
    nw = ops.NativeWeights(torch.from_numpy(oracle.pack(W).view(np.int32)).to(cuda), N)
    x = rng.standard_normal((M, K)).astype(np.float32) * np.float32(10.0) ** (np.arange(M)[:, None] // 8 % 9 - 4).astype(np.float32)
    want, size = torch.from_numpy(x.astype(np.float64) @ W.T), torch.from_numpy(np.abs(x).astype(np.float64).sum(1, keepdims=True))
    y = ops.ternary_linear(torch.from_numpy(x).to(cuda), nw).double().cpu()
    assert torch.all((y - want).abs() <= size * (2.0 ** -22 + (K / 16 + 64) * 2.0 ** -24))
