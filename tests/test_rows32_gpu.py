"""Up to sixteen short fp32 rows, split into fp16 terms by the workgroups that multiply them (rows32.hip)."""
import ctypes

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _check(cuda, oracle, M, K, N):
    from tmq_amd import ops, _capi
    print("rows32", M, K, N, flush=True)
    lib = _capi.load()
    rng = np.random.default_rng(M * 1000003 + K * 1009 + N)
    W = rng.integers(-1, 2, size=(N, K)).astype(np.float32)
    nw = ops.NativeWeights(torch.from_numpy(oracle.pack(W).view(np.int32)).to(cuda), N)
    # every row a magnitude of its own, one of zeros among them
    x = rng.standard_normal((M, K)).astype(np.float32) * np.float32(10.0) ** rng.integers(-30, 30, size=(M, 1)).astype(np.float32)
    if M > 2:
        x[M - 2] = 0.0
    tx = torch.from_numpy(x).to(cuda)
    scale, bias = (0.5 + rng.random(N)).astype(np.float32), rng.standard_normal(N).astype(np.float32)
    res = rng.standard_normal((M, N)).astype(np.float32)
    t = lambda a: torch.from_numpy(a).to(cuda)
    assert lib.tmq_fp32_rows_one_launch(ops.ptr(tx), M, K, N) == 1
    want = x.astype(np.float64) @ W.astype(np.float64).T
    # 22 bits a value, and a rounding for each of a wavefront's products (32 indices each), the eight wavefronts' sums, the
    # pair's and the 32 additions inside a product, each of the largest partial sum at most
    size = np.abs(x.astype(np.float64)).sum(1, keepdims=True)
    bound = size * (2.0 ** -22 + (2 * -(-K // 512) + 8 + 2 + 33) * 2.0 ** -24)
    y = ops.ternary_linear(tx, nw)
    assert np.all(np.abs(y.cpu().numpy() - want) <= bound + 1e-45)
    assert torch.equal(ops.ternary_linear(tx, nw), y)
    # the epilogue, through the C entry with and without a workspace (not used)
    ts, tb, tr = t(scale), t(bias), t(res)
    ep = _capi.Epilogue(ops.ptr(ts), ops.ptr(tb), ops.ptr(tr), 1, _capi.F32)
    ws = torch.empty(max(16, lib.tmq_ternary_linear_workspace_bytes(_capi.F32, M, K, N)), dtype=torch.uint8, device=cuda)
    full = np.maximum(want * scale + bias + res, 0)
    tol = bound * scale * 1.01 + np.abs(want * scale) * 2.0 ** -22 + 1e-6
    for wptr, n in ((ops.ptr(ws), ws.numel()), (None, 0)):
        y2 = torch.full_like(y, float("nan"))
        assert lib.tmq_ternary_linear_ws(ops.ptr(tx), _capi.F32, M, K, ops.ptr(nw.buf), N, ctypes.byref(ep), ops.ptr(y2), wptr, n, None) == 0
        torch.cuda.synchronize()
        assert np.all(np.abs(y2.cpu().numpy() - full) <= tol)
    small = ops.ternary_linear(tx * 0 + 1, nw, ts, tb, residual=tr.half(), out_dtype=torch.float16).float().cpu().numpy()
    ref = W.astype(np.float64).sum(1)[None] * scale + bias + res.astype(np.float16)
    assert np.all(np.abs(small - ref) <= np.abs(ref) * 2.0 ** -10 + 1e-3)


@pytest.mark.parametrize("M", [1, 2, 3, 4, 5, 8, 9, 15, 16])
@pytest.mark.parametrize("K,N", [(1, 1), (7, 15), (63, 16), (64, 17), (65, 260), (511, 33), (513, 4097), (1000, 3000), (1025, 8195), (2047, 30), (2048, 300)])
def test_rows_against_fp64(cuda, oracle, M, K, N):
    _check(cuda, oracle, M, K, N)


@pytest.mark.parametrize("M,K,N", [(1, 4095, 100), (3, 4096, 4096), (5, 2049, 4095), (8, 4096, 17), (2, 129, 20000), (12, 200, 33000)])
def test_longest_and_widest(cuda, oracle, M, K, N):
    _check(cuda, oracle, M, K, N)


def test_where_the_lines_lie(cuda, oracle):
    from tmq_amd import _capi
    one = _capi.load().tmq_fp32_rows_one_launch
    assert [one(None, M, 2048, 512) for M in (8, 9, 16, 17)] == [1, 1, 1, 0]
    assert [one(None, 8, K, 512) for K in (2048, 2049, 4096, 4097)] == [1, 1, 1, 0]
    assert [one(None, 16, K, 512) for K in (2048, 2049)] == [1, 0]
    assert [one(None, 3, 4096, N) for N in (4096, 4097)] == [1, 0]
    assert [one(None, 3, 2048, N) for N in (12288, 12289)] == [1, 0]
    assert [one(None, 9, 2048, N) for N in (16384, 16385)] == [1, 0]
    assert one(None, 0, 512, 512) == 0 and one(ctypes.c_void_p(4), 3, 512, 512) == 0


@pytest.mark.parametrize("M", [5, 12])
def test_infinities_and_nan_stay_in_their_row(cuda, oracle, M):
    from tmq_amd import ops
    K, N = 777, 130
    rng = np.random.default_rng(M)
    W = rng.integers(-1, 2, size=(N, K)).astype(np.float32)
    nw = ops.NativeWeights(torch.from_numpy(oracle.pack(W).view(np.int32)).to(cuda), N)
    x = rng.standard_normal((M, K)).astype(np.float32)
    clean = ops.ternary_linear(torch.from_numpy(x).to(cuda), nw).cpu()
    x[1, 300], x[3, 776] = np.nan, np.inf
    y = ops.ternary_linear(torch.from_numpy(x).to(cuda), nw).cpu()
    keep = [m for m in range(M) if m not in (1, 3)]
    assert torch.equal(y[keep], clean[keep])
    assert torch.isnan(y[1]).all() and not torch.isfinite(y[3]).any()


@pytest.mark.parametrize("M,K,N", [(16, 40, 33000), (4, 1100, 17000)])
def test_widest_layers_without_a_workspace_take_rows_of_any_magnitude(cuda, oracle, M, K, N):
    """tmq_fp32_rows_one_launch prefers the workspace there; the call without one still scales the rows itself."""
    from tmq_amd import ops, _capi
    lib = _capi.load()
    rng = np.random.default_rng(M)
    W = rng.integers(-1, 2, size=(N, K)).astype(np.float32)
    nw = ops.NativeWeights(torch.from_numpy(oracle.pack(W).view(np.int32)).to(cuda), N)
    x = rng.standard_normal((M, K)).astype(np.float32) * np.float32(10.0) ** rng.integers(-30, 30, size=(M, 1)).astype(np.float32)
    tx = torch.from_numpy(x).to(cuda)
    assert lib.tmq_fp32_rows_one_launch(ops.ptr(tx), M, K, N) == 0
    want = x.astype(np.float64) @ W.astype(np.float64).T
    bound = np.abs(x.astype(np.float64)).sum(1, keepdims=True) * (2.0 ** -22 + (2 * -(-K // 512) + 8 + 2 + 33) * 2.0 ** -24)
    y = torch.full((M, N), float("nan"), device=cuda)
    assert lib.tmq_ternary_linear(ops.ptr(tx), _capi.F32, M, K, ops.ptr(nw.buf), N, None, ops.ptr(y), None) == 0
    torch.cuda.synchronize()
    assert np.all(np.abs(y.cpu().numpy() - want) <= bound + 1e-45)
    # with the workspace: the rows' own powers of two as well, 22 bits a value, sums over up to K / 32 products
    z = ops.ternary_linear(tx, nw)
    assert np.all(np.abs(z.cpu().numpy() - want) <= 2 * bound + 1e-45)
