"""The opening of a network on fp32 images in one kernel behind the scan for the largest magnitude: the prescale, the
rounding to fp16 and the constants are those of tmq_f32_to_f16_prescaled followed by the fp16 opening, so the two agree bit
for bit; both heights of a patch (3 pooled rows up to 768 patches, 7 beyond) and their ragged last rows."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


def _layer(cuda, C, N, k, pad, seed):
    import tmq_amd as t
    torch.manual_seed(seed)
    net = torch.nn.Sequential(torch.nn.Conv2d(C, N, k, 2, pad, bias=False))
    ctrl = t.QuantizationControl()
    t.quantize_model(net, ctrl)
    net.to(cuda).eval()
    ctrl.quantize()
    t.compressed_state_dict(net, strong=False)
    return net[0]


# one image (3 pooled rows a patch; 56 = 18 * 3 + 2), seven (7 rows), patches cut at the right and lower edge, one to four
# planes, windows whose reduction ends inside a matrix step (k = 3, 5), a batch with partial maxima of its full count
@pytest.mark.parametrize("B,C,H,W,N,k,pad", [(1, 3, 224, 224, 64, 7, 3), (7, 3, 224, 216, 64, 7, 3), (2, 3, 33, 48, 64, 7, 3), (3, 1, 20, 24, 16, 5, 2),
                                             (2, 4, 17, 20, 40, 3, 1), (1, 2, 9, 12, 8, 7, 3), (33, 3, 64, 60, 32, 3, 0), (40, 3, 224, 224, 24, 7, 3)])
@pytest.mark.parametrize("values", ["normal", "large", "tiny", "special"])
def test_fp32_opening_equals_prescale_then_opening(cuda, B, C, H, W, N, k, pad, values):
    from tmq_amd import ops
    conv = _layer(cuda, C, N, k, pad, B + C + H)
    x = torch.randn((B, C, H, W), device=cuda)
    if values == "large":
        x *= 3e30
    elif values == "tiny":
        x *= 1e-30
    elif values == "special":        # out of the maximum, and what they touch stays what the two calls make of it
        x[0, 0, 0, 0], x[-1, -1, -1, -1], x[0, 0, H // 2, W // 2] = float("inf"), float("-inf"), float("nan")
    nw, kxs, pl, pr = conv._superpixel_plan(x)
    scale, bias = torch.rand(N, device=cuda) - 0.3, torch.randn(N, device=cuda)
    form = ((2, 1), ((pad, pad), (pl, pr)), 1)
    for sc in (scale, None):
        h, adjusted = ops.f32_to_f16_prescaled(x, sc, N)
        xs = ops.nchw_to_nhwc4(h).view(B, H, W // 2, 8).permute(0, 3, 1, 2)
        want = F.max_pool2d(F.relu(ops.ternary_conv2d(xs, nw, *form, scale=adjusted, bias=bias, out_dtype=torch.float16)), 3, 2, 1)
        planar = ops.ternary_conv2d_relu_maxpool_planar(h, nw, *form, adjusted, bias)
        got = ops.ternary_conv2d_relu_maxpool_planar(x, nw, *form, sc, bias, prescale=True)
        assert got.dtype == torch.float16 and torch.equal(got.view(torch.int16), planar.view(torch.int16))
        if values != "special":      # (a max-pool on its own treats a NaN differently)
            assert torch.equal(got, want)
    # rows that 8-byte loads cannot take, and a view that is not contiguous: converted first, the same bits
    buf = torch.empty(x.numel() + 1, device=cuda)
    odd = buf[1:].view(x.shape)
    odd.copy_(x)
    wide = torch.zeros((B, C, H, W + 4), device=cuda)
    wide[..., 2:W + 2] = x
    for other in (odd, wide[..., 2:W + 2]):
        again = ops.ternary_conv2d_relu_maxpool_planar(other, nw, *form, None, bias, prescale=True)
        assert torch.equal(again.view(torch.int16), got.view(torch.int16))


def test_fp32_opening_in_a_graph(cuda):
    from tmq_amd import ops
    conv = _layer(cuda, 3, 64, 7, 3, 1)
    x = torch.randn((2, 3, 96, 96), device=cuda)
    nw, kxs, pl, pr = conv._superpixel_plan(x)
    form = ((2, 1), ((3, 3), (pl, pr)), 1)
    call = lambda: ops.ternary_conv2d_relu_maxpool_planar(x, nw, *form, prescale=True)
    call()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = call()
    for factor in (1.0, 1e6, 1e-9):
        x.copy_(torch.randn_like(x) * factor)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, call())


# more patches than the fp32 form is taken for: converted first, the same bits
@pytest.mark.parametrize("planes,stride,B", [(1, (2, 2), 80), (2, (1, 2), 40), (4, (1, 2), 27)])
def test_many_patches_are_converted_first(cuda, planes, stride, B):
    import tmq_amd as t
    from tmq_amd import ops
    torch.manual_seed(planes)
    net = torch.nn.Sequential(torch.nn.Conv2d(planes, 8, 3, stride, 1, bias=False))
    ctrl = t.QuantizationControl()
    t.quantize_model(net, ctrl)
    net.to(cuda).eval()
    ctrl.quantize()
    t.compressed_state_dict(net, strong=False)
    x = torch.randn((B, planes, 256, 304), device=cuda) * 1e5
    nw, kxs, pl, pr = net[0]._superpixel_plan(x)
    form = ((stride[0], 1), ((1, 1), (pl, pr)), 1)
    h, adjusted = ops.f32_to_f16_prescaled(x, None, 8)
    want = ops.ternary_conv2d_relu_maxpool_planar(h, nw, *form, adjusted)
    got = ops.ternary_conv2d_relu_maxpool_planar(x, nw, *form, prescale=True)
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))
