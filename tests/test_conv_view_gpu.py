"""tmq_ternary_conv2d_view: a convolution whose output positions are scattered into a strided NHWC destination
(how a transposed convolution with groups == 1 is written in one pass, tmq/tmq.py:1007-1042 plans GEMM + F.fold).

Bar: bit-identical to tmq_ternary_conv2d followed by a strided copy of the kept window (the same kernel computes the
same sums; only the addresses of its stores change), every element outside the destination view untouched, for every
kernel family a convolution can take (direct-to-LDS tiles on 64-channel and few-channel inputs, register-staged tiles,
the eight-wavefront 64 x 256 tiles, the split-reduction kernel), fp16 and fp32 outputs, residual and ReLU; and
ConvTranspose2d at sizes beyond the exact small cases of test_dwconv_gpu.py against F.conv_transpose2d (fp64 and the
layer's own float forward).
"""
import ctypes

import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


# (B, C, H, W, N, k, pad, dil): which kernel the dispatch of tmq_ternary_conv2d picks for it
CASES = [
    (4, 64, 20, 20, 64, 3, 1, 1),       # tile_dma_kernel, ConvLoader64, 64 x 64 tiles
    (2, 64, 40, 40, 192, 3, 1, 1),      # 129 .. 256 channels over >= 8192 positions: tile_solo_kernel 64 x 256
    (3, 16, 17, 19, 40, 3, 1, 1),       # few-channel loader
    (2, 12, 9, 11, 24, (3, 2), (1, 0), 1),   # register-staged loader, 8-byte aligned pixels
    (2, 5, 9, 11, 7, 3, 1, 1),          # scalar loader, odd channel counts (scalar stores)
    (2, 128, 14, 14, 128, 3, 1, 1),     # split reduction inside the workgroup (mid_kernel, ConvRows)
    (1, 256, 7, 7, 512, 3, 1, 1),       # the same with four wavefronts per tile
    (2, 64, 12, 12, 64, 2, 0, 2),       # dilation
]


@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_view_equals_dense_then_copy(cuda, case, dtype):
    from tmq_amd import ops
    B, C, H, W, N, k, pad, dil = case
    print("conv view", case, dtype, flush=True)
    pair = lambda v: tuple(v) if isinstance(v, (tuple, list)) else (v, v)
    g = torch.Generator(device=cuda).manual_seed(C * 1000 + N)
    Wt = torch.randint(-1, 2, (N, C) + pair(k), device=cuda, generator=g).float()
    nw = ops.NativeWeights(ops.compactify_ternary(Wt), N, conv_kernel=pair(k))
    x = torch.randn((B, C, H, W), device=cuda, generator=g).half().contiguous(memory_format=torch.channels_last)
    scale = (torch.rand(N, device=cuda, generator=g) + 0.5) * 0.05
    bias = torch.randn(N, device=cuda, generator=g)
    dense = ops.ternary_conv2d(x, nw, 1, pad, dil, scale, bias, out_dtype=dtype)
    ho, wo = dense.shape[2:]
    # the window of the computed grid that is kept, and where it lands in a larger interleaved tensor
    for (h0, w0, hc, wc), (sy, sx), (oy, ox) in [((0, 0, ho, wo), (2, 2), (1, 0)), ((1, 2, ho - 2, wo - 3), (3, 2), (2, 1)),
                                                 ((0, 0, ho, wo), (1, 1), (0, 0))]:
        big = torch.full((B, N, oy + sy * hc + 1, ox + sx * wc + 2), 7.0, dtype=dtype, device=cuda).contiguous(memory_format=torch.channels_last)
        want = big.clone()
        want[:, :, oy:oy + sy * hc:sy, ox:ox + sx * wc:sx] = dense[:, :, h0:h0 + hc, w0:w0 + wc]
        target = big[:, :, oy:oy + sy * hc:sy, ox:ox + sx * wc:sx]
        assert target.shape[2:] == (hc, wc)
        ops.ternary_conv2d_into(target, x, nw, 1, pad, dil, scale, bias, first=(h0, w0))
        assert torch.equal(big, want), (case, (h0, w0, hc, wc), (sy, sx))
    # residual (read at the destination's own offsets) and ReLU
    res_big = torch.randn((B, N, 2 * ho, 2 * wo), device=cuda, generator=g).to(dtype).contiguous(memory_format=torch.channels_last)
    res = res_big[:, :, 1::2, 0::2]
    dense_r = ops.ternary_conv2d(x, nw, 1, pad, dil, scale, bias, residual=res.contiguous(memory_format=torch.channels_last),
                                 relu=True, out_dtype=dtype)
    big = torch.zeros_like(res_big)
    ops.ternary_conv2d_into(big[:, :, 1::2, 0::2], x, nw, 1, pad, dil, scale, bias, residual=res, relu=True)
    assert torch.equal(big[:, :, 1::2, 0::2], dense_r)
    assert int(big[:, :, 0::2].count_nonzero()) == 0 and int(big[:, :, :, 1::2].count_nonzero()) == 0


def test_view_in_place_residual_and_argument_checks(cuda):
    """The residual may be the destination itself (accumulating phases); malformed views are refused."""
    from tmq_amd import ops, _capi
    g = torch.Generator(device=cuda).manual_seed(5)
    Wt = torch.randint(-1, 2, (64, 64, 3, 3), device=cuda, generator=g).float()
    nw = ops.NativeWeights(ops.compactify_ternary(Wt), 64, conv_kernel=(3, 3))
    x = torch.randint(-3, 4, (2, 64, 10, 10), device=cuda, generator=g).half().contiguous(memory_format=torch.channels_last)
    big = torch.randint(-5, 6, (2, 64, 20, 20), device=cuda, generator=g).float().contiguous(memory_format=torch.channels_last)
    want = big.clone()
    want[:, :, 0::2, 1::2] += F.conv2d(x.float(), Wt, None, 1, 1)
    ops.ternary_conv2d_into(big[:, :, 0::2, 1::2], x, nw, 1, 1, 1, residual=big[:, :, 0::2, 1::2])
    assert torch.equal(big, want)
    with pytest.raises(RuntimeError):
        ops.ternary_conv2d_into(big[:, :32, 0::2, 1::2], x, nw, 1, 1, 1)                 # channel slice: pixels are not N wide
    with pytest.raises(RuntimeError):
        ops.ternary_conv2d_into(big.contiguous()[:, :, 0::2, 1::2], x, nw, 1, 1, 1)      # NCHW memory
    lib = _capi.load()
    shp = _capi.ConvShape(2, 64, 10, 10, 64, 3, 3, 1, 1, 1, 1, 1, 1, 1, 1)
    ep = _capi.Epilogue(None, None, None, 0, _capi.F32)
    for bad in [_capi.OutputView(0, 0, 11, 10, 400, 40, 2), _capi.OutputView(-1, 0, 5, 5, 400, 40, 2),
                _capi.OutputView(3, 0, 8, 10, 400, 40, 2), _capi.OutputView(0, 0, 10, 10, -1, 40, 2)]:
        assert lib.tmq_ternary_conv2d_view(ops.ptr(x), ctypes.byref(shp), ops.ptr(nw.buf), ctypes.byref(ep), ops.ptr(big),
                                           ctypes.byref(bad), None) == -1        # TMQ_ERR_INVALID_ARG
    before = big.clone()                                                                # an empty window: nothing is written
    assert lib.tmq_ternary_conv2d_view(ops.ptr(x), ctypes.byref(shp), ops.ptr(nw.buf), ctypes.byref(ep), ops.ptr(big),
                                       ctypes.byref(_capi.OutputView(0, 0, 0, 10, 400, 40, 2)), None) == 0
    torch.cuda.synchronize()
    assert torch.equal(big, before)


@pytest.mark.parametrize("cin,cout,k,stride,pad,opad,hw,batch", [
    (64, 64, 4, 2, 1, 0, (32, 32), 8),         # the usual decoder layer at a size that fills the chip
    (128, 64, 3, 2, 1, 1, (16, 16), 4),        # odd kernel: phases with 2 x 2, 2 x 1, 1 x 2 and 1 x 1 taps
    (256, 128, 2, 2, 0, 0, (14, 14), 2),       # non-overlapping up-sampling: every phase a 1 x 1 convolution
    (64, 192, 5, 3, 2, 1, (20, 24), 4)])       # stride 3, 129 .. 256 output channels
def test_transposed_layer_one_pass(cuda, cin, cout, k, stride, pad, opad, hw, batch):
    import tmq_amd as t
    torch.manual_seed(cin + cout + k)
    net = torch.nn.Sequential(torch.nn.ConvTranspose2d(cin, cout, k, stride, pad, output_padding=opad, bias=True))
    ctrl = t.QuantizationControl()
    t.quantize_model(net, ctrl)
    net.to(cuda).eval()
    ctrl.quantize()
    layer = net[0]
    Wt = layer.weight.data.clone()
    assert set(Wt.unique().tolist()) <= {-1.0, 0.0, 1.0}
    x = torch.randn((batch, cin) + hw, device=cuda)
    x16 = x.half()
    with torch.no_grad():
        ref = net(x16.float()).double()                    # the layer's own float forward on the ternarised weights
    plain = F.conv_transpose2d(x16.double(), Wt.double(), layer.bias.data.double(), stride, pad, opad)
    assert ((ref - plain).abs().max() / plain.abs().max()).item() <= 2e-5
    t.compressed_state_dict(net, strong=False)
    assert layer.weight.dtype == torch.int32
    launches = []
    from tmq_amd import ops
    orig = ops.ternary_conv2d_into

    def counted(*a, **kw):
        launches.append(1)
        return orig(*a, **kw)

    ops.ternary_conv2d_into = counted
    try:
        got = net(x16)
    finally:
        ops.ternary_conv2d_into = orig
    sy = stride if isinstance(stride, int) else stride[0]
    assert 1 <= len(launches) <= sy * sy                   # one launch per phase, nothing else
    assert got.shape == ref.shape
    err = ((got.double() - ref).abs().max() / ref.abs().max()).item()
    assert err <= 2e-5, err


@pytest.mark.parametrize("cin,cout,k,stride,pad,hw,batch", [
    (64, 64, 4, 2, 1, (33, 18), 3),            # one launch of four phases; 64 x 64 tiles, ragged last tile
    (64, 130, 3, 2, 1, (70, 66), 2),           # 128 x 128 tiles, phases of 2 x 2, 2 x 1, 1 x 2 and 1 x 1 taps, a third column tile
    (128, 66, 5, 3, 2, (9, 11), 2),            # nine phases: three launches
    (32, 40, 4, 2, 1, (17, 9), 2), (8, 7, 4, 2, 1, (9, 9), 2),       # the few-channel loader
    (24, 72, 4, 2, 1, (60, 60), 2), (104, 16, 3, 2, 1, (13, 7), 1),  # register-staged loaders: whole 16-byte chunks,
    (100, 64, 4, 2, 1, (14, 15), 2), (5, 9, 4, 2, 1, (7, 8), 2),     # halves of 8 bytes, single elements
    (300, 20, 4, 2, 1, (6, 5), 1)])            # a reduction long enough for the deeper prefetch
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_phases_in_one_launch_equal_one_launch_each(cuda, cin, cout, k, stride, pad, hw, batch, dtype):
    """ops.ternary_conv2d_into(phases=...): every phase of a transposed convolution written by the shared launch equals the
    same phase written by a launch of its own (small integers: exact in either summation order), with residual and ReLU."""
    import copy
    import tmq_amd as t
    from tmq_amd import ops
    torch.manual_seed(cin * 100 + cout)
    net = torch.nn.Sequential(torch.nn.ConvTranspose2d(cin, cout, k, stride, pad, bias=True))
    t.quantize_model(net, t.QuantizationControl())
    net.to(cuda).eval()
    net[0].weight.data = torch.randint(-1, 2, net[0].weight.shape, device=cuda).float()
    net[0].bias.data = torch.randint(-4, 5, (cout,), device=cuda).float()
    t.compressed_state_dict(net)
    layer = net[0]
    x = torch.randint(-3, 4, (batch, cin) + hw, device=cuda).half().contiguous(memory_format=torch.channels_last)
    want = F.conv_transpose2d(x.cpu().float(), ops.expand_ternary(layer.weight.data, layer.original_shape).cpu(),
                              layer.bias.data.cpu(), stride, pad).to(dtype)
    prev = t.set_compact_output_dtype(dtype)
    try:
        got = net(x)
        again = copy.deepcopy(net)(x)                       # a copy plans for its own weights
        net(x[:, :, :5, :4])                                # another shape in between
        assert torch.equal(got.cpu(), want) and torch.equal(again, got) and torch.equal(net(x), got)
    finally:
        t.set_compact_output_dtype(prev)
    plan = layer._phases[2]
    res = torch.randint(-9, 10, got.shape, device=cuda).to(dtype).contiguous(memory_format=torch.channels_last)
    one = ops.ternary_conv2d_into(torch.empty_like(res), x, None, residual=res, relu=True, phases=plan)
    each = torch.empty_like(res)
    for nw, padding, dil, first, (o0, p0), (sy, sx), _ in plan.parts:
        ops.ternary_conv2d_into(each[:, :, o0::sy, p0::sx], x, nw, 1, padding, dil, residual=res[:, :, o0::sy, p0::sx], relu=True, first=first)
    assert torch.equal(one, each)
    with pytest.raises(RuntimeError):
        ops.ternary_conv2d_into(each[:, :, :-1], x, None, phases=plan)


@pytest.mark.parametrize("B,C,hw,N,k", [
    (1, 64, (41, 50), 70, 1),          # short reduction: 64 x 128 tiles, a ragged last tile in rows and columns
    (1, 64, (116, 127), 200, 1),       # 462 of them in two 128s: 64 x 256
    (1, 128, (190, 100), 300, 1),      # 891 in three, N no multiple of 8: the general tiles
    (1, 64, (86, 96), 128, 3),         # 129 tiles at K = 576, where the split reduction ends: 64 x 128 solo
    (1, 64, (129, 128), 100, 3),       # 258 tiles, N <= 128: dma at K = 576 ...
    (1, 128, (129, 128), 128, 3),      # ... solo at K = 1152
    (1, 128, (96, 121), 130, 3),       # 129 .. 256 columns, 364 tiles: 64 x 128 solo
    (1, 64, (82, 81), 300, 3),         # three 128s, short of K = 1024: dma ...
    (1, 64, (107, 109), 300, 3),       # ... for any number of tiles
    (1, 64, (71, 73), 400, 3),         # and four
    (2, 64, (97, 95), 32, 3),          # at most 32 columns: 128 x 32 tiles, a ragged last one, direct loads ...
    (3, 16, (31, 33), 17, 5), (1, 104, (40, 41), 24, 3),     # ... of few channels, through registers
    (1, 136, (19, 21), 30, 3), (2, 17, (15, 16), 5, 3)])     # (reduction of 1224: deeper prefetch; single elements)
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_wide_tiles_at_their_edges(cuda, B, C, hw, N, k, dtype):
    """Convolutions on the tiles of 64 x 128 and 64 x 256 (more than 64 outputs) and 128 x 32 (at most 32), the rules of
    their choice, against F.conv2d: small integers, so every sum is exact (fp16 results: below 2^11)."""
    from tmq_amd import ops
    g = torch.Generator(device=cuda).manual_seed(C + N + k)
    Wt = torch.randint(-1, 2, (N, C, k, k), device=cuda, generator=g).float()
    nw = ops.NativeWeights(ops.compactify_ternary(Wt), N, conv_kernel=(k, k))
    x = torch.randint(-2, 3, (B, C) + hw, device=cuda, generator=g).half().contiguous(memory_format=torch.channels_last)
    bias = torch.randint(-4, 5, (N,), device=cuda, generator=g).float()
    res = torch.randint(-9, 10, (B, N) + hw, device=cuda, generator=g).to(dtype).contiguous(memory_format=torch.channels_last)
    want = F.conv2d(x.cpu().float(), Wt.cpu(), bias.cpu(), 1, k // 2)
    assert want.abs().max() < 2000
    assert torch.equal(ops.ternary_conv2d(x, nw, 1, k // 2, 1, bias=bias, out_dtype=dtype).cpu().float(), want)
    got = ops.ternary_conv2d(x, nw, 1, k // 2, 1, bias=bias, residual=res, relu=True, out_dtype=dtype)
    assert torch.equal(got.cpu().float(), torch.relu(want + res.cpu().float()))


def test_transposed_layer_follows_a_change_of_padding(cuda):
    """Padding and output padding set anew on a layer that has planned its phases, the output keeping its size."""
    import tmq_amd as t
    torch.manual_seed(5)
    net = torch.nn.Sequential(torch.nn.ConvTranspose2d(8, 7, 3, 3, 0, bias=False))
    t.quantize_model(net, t.QuantizationControl())
    net.to(cuda).eval()
    w = torch.randint(-1, 2, net[0].weight.shape, device=cuda).float()
    net[0].weight.data = w
    t.compressed_state_dict(net)
    x = torch.randint(-3, 4, (2, 8, 8, 8), device=cuda).half()
    for pad, opad in ((0, 0), (1, 2), (0, 0)):
        net[0].padding, net[0].output_padding = (pad, pad), (opad, opad)
        assert torch.equal(net(x).cpu(), F.conv_transpose2d(x.cpu().float(), w.cpu(), None, 3, pad, opad))


@pytest.mark.parametrize("cin,cout,k,stride,pad,hw,batch", [
    (64, 40, 3, 1, 1, (9, 7), 2), (24, 33, 2, 1, 0, (6, 9), 1),            # one phase: an ordinary convolution
    (512, 48, (6, 6), (2, 2), (2, 2), (5, 6), 1),                              # four phases of few tiles and long reductions: one by one
    (128, 70, (2, 4), (1, 2), (0, 1), (6, 5), 1), (64, 34, (1, 2), (1, 2), 0, (6, 5), 3),   # two, either way
    (64, 30, (3, 3), (3, 3), 0, (6, 5), 1)])                                # nine: two groups of four, the last one alone
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_phases_alone_or_of_long_reductions_take_their_own_launches(cuda, cin, cout, k, stride, pad, hw, batch, dtype):
    """Each side of the rule that sends the phases of a transposed convolution through one launch or through the route of an
    ordinary convolution, with residual and ReLU, against F.conv_transpose2d (small integers: exact)."""
    import tmq_amd as t
    from tmq_amd import ops
    torch.manual_seed(cin + cout)
    net = torch.nn.Sequential(torch.nn.ConvTranspose2d(cin, cout, k, stride, pad, bias=True))
    t.quantize_model(net, t.QuantizationControl())
    net.to(cuda).eval()
    net[0].weight.data = torch.randint(-1, 2, net[0].weight.shape, device=cuda).float()
    net[0].bias.data = torch.randint(-4, 5, (cout,), device=cuda).float()
    t.compressed_state_dict(net)
    x = torch.randint(-2, 3, (batch, cin) + hw, device=cuda).half().contiguous(memory_format=torch.channels_last)
    want = F.conv_transpose2d(x.cpu().float(), ops.expand_ternary(net[0].weight.data, net[0].original_shape).cpu(),
                              net[0].bias.data.cpu(), stride, pad)
    assert want.abs().max() < 2000
    prev = t.set_compact_output_dtype(dtype)
    try:
        assert torch.equal(net(x).cpu(), want.to(dtype))
    finally:
        t.set_compact_output_dtype(prev)
    res = torch.randint(-9, 10, want.shape, device=cuda).to(dtype).contiguous(memory_format=torch.channels_last)
    got = ops.ternary_conv2d_into(torch.empty_like(res), x, None, bias=net[0].bias.data, residual=res, relu=True, phases=net[0]._phases[2])
    assert torch.equal(got.cpu(), torch.relu(want + res.cpu().float()).to(dtype))


@pytest.mark.parametrize("B,C,hw,N,k", [
    (1, 128, (82, 81), 300, 3),        # three 128s from K = 1024 on: 312 tiles, solo
    (1, 128, (70, 73), 500, 3),        # four: 320
    (1, 128, (110, 100), 504, 3),      # 688
    (1, 128, (120, 116), 400, 3),      # 872: the general tiles
    (1, 128, (150, 151), 264, 3),      # three, 1062: dma
    (1, 64, (131, 141), 250, 3),       # two, 578: 64 x 256 solo, at K = 576 ...
    (1, 128, (131, 141), 250, 3),      # ... and 1152
    (1, 128, (112, 113), 104, 3),      # one, 198, where the split reduction ends: solo
    (1, 64, (62, 64), 1032, 1),        # nine 128s: dma
    (1, 128, (81, 83), 170, 1),        # two, 212: dma
    (1, 128, (50, 51), 1024, 3),       # eight, 320: solo
    (1, 64, (40, 41), 1033, 1),        # (an odd width)
    (1, 64, (23, 25), 2050, 1),        # beyond 2048: the general tiles
    (1, 64, (313, 315), 76, 1)])       # 1541 of one 128: dma
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_wide_tiles_by_rows_reduction_and_width(cuda, B, C, hw, N, k, dtype):
    """The other lines of that choice, tile counts that are no multiple of 8 among them (their order over the XCDs)."""
    test_wide_tiles_at_their_edges(cuda, B, C, hw, N, k, dtype)


@pytest.mark.parametrize("M,K,N", [(16448, 4096, 24), (16448, 4032, 30), (129, 4100, 7)])
def test_few_outputs_on_either_tile(cuda, M, K, N):
    """Dense rows into at most 32 outputs below and from K = 4096 on (128 x 32 and 64 x 64 tiles), and single elements: exact."""
    from tmq_amd import ops
    g = torch.Generator(device=cuda).manual_seed(M + K)
    Wt = torch.randint(-1, 2, (N, K), device=cuda, generator=g).float()
    x = torch.randint(-2, 3, (M, K), device=cuda, generator=g).half()
    nw = ops.NativeWeights(ops.compactify_ternary(Wt), N)
    assert torch.equal(ops.ternary_linear(x, nw).cpu(), (x.cpu().float() @ Wt.cpu().t()))


@pytest.mark.parametrize("B,C,hw,N", [(1, 34, (99, 28), 14), (1, 36, (99, 28), 14), (2, 134, (9, 28), 31)])
def test_few_outputs_of_odd_channels_on_either_tile(cuda, B, C, hw, N):
    """Convolutions into at most 32 outputs that read single elements (64 x 64 tiles) and halves of 8 bytes (128 x 32)."""
    test_wide_tiles_at_their_edges(cuda, B, C, hw, N, 3, torch.float32)
