"""Which kernel a convolution is sent to (tmq_ternary_conv2d_kernel, host only)."""
import ctypes

import pytest

TILES, SPLIT, PATCH = 0, 1, 2


def kernel_of(B, C, H, W, N, k, pad, d=1, s=1, f16=True):
    """k: (ky, kx); pad: ((top, bottom), (left, right)) or one number."""
    from tmq_amd import _capi
    (pt, pb), (pl, pr) = pad if isinstance(pad, tuple) else ((pad, pad), (pad, pad))
    shape = _capi.ConvShape(B, C, H, W, N, k[0], k[1], s, s, pt, pl, d, d, pb, pr)
    return _capi.load().tmq_ternary_conv2d_kernel(ctypes.byref(shape), _capi.F16 if f16 else _capi.F32)


# the largest distance of a tap in the padded image, 2 d (14 + d) + 2 d, passes 2^31 from d = 32761 on
@pytest.mark.parametrize("d", [1000, 30000, 32759, 32760, 32768, 33000, 40000, 46341, 65536])
def test_far_taps_do_not_fit_a_patch(d):
    assert kernel_of(64, 256, 14, 14, 256, (3, 3), 1) == PATCH
    assert kernel_of(64, 256, 14, 14, 256, (3, 3), d, d) != PATCH
    assert kernel_of(64, 256, 14, 14, 256, (1, 9), ((0, 0), (4 * d, 4 * d)), d) != PATCH
    assert kernel_of(64, 256, 14, 14, 256, (9, 1), ((4 * d, 4 * d), (0, 0)), d) != PATCH


# half of such workgroups' reduction, and at most 64 outputs are two rounds of the chip where the plan counts one
@pytest.mark.parametrize("B,H,W,N", [(64, 28, 28, 128), (32, 56, 56, 64), (162, 27, 25, 64), (32, 83, 10, 244), (28, 109, 3, 640)])
@pytest.mark.parametrize("f16", [False, True])
def test_128_channels_stay_out_of_patches(B, H, W, N, f16):
    assert kernel_of(B, 128, H, W, N, (3, 3), 1, f16=f16) != PATCH


# 512 channels: at most 256 tiles of 64 x 64, then more of them (0.57 to 0.59 of a round of units)
def test_one_round_of_tiles_stays_out_of_patches():
    for B, H, W, N, pad in [(47, 16, 8, 448, 0), (25, 23, 3, 576, 1), (40, 10, 5, 512, 1), (31, 7, 8, 572, 1)]:
        assert kernel_of(B, 512, H, W, N, (3, 3), pad, f16=False) != PATCH
    for B, H, W, N in [(32, 12, 6, 456), (44, 7, 6, 576), (20, 35, 4, 384)]:
        assert kernel_of(B, 512, H, W, N, (3, 3), 1) == PATCH


def test_refuses_what_the_convolution_refuses():
    from tmq_amd import _capi
    assert kernel_of(1, 64, 3, 3, 64, (5, 5), 0) == -1 and kernel_of(1, 64, 0, 3, 64, (1, 1), 0) == -1
    assert _capi.load().tmq_ternary_conv2d_kernel(None, _capi.F32) == -1
    assert kernel_of(0, 64, 8, 8, 64, (3, 3), 1) >= 0          # an empty batch is nothing to launch


def test_fp32_opening_leaves_many_patches_to_the_conversion():
    from tmq_amd import _capi

    def pays(planes, sy, B, size=224):
        # a 7 x 7 opening of horizontal stride 2 over super-pixels: 8 x 7 patches a 224 x 224 image at vertical stride 2, 16 x 7 at 1
        shape = _capi.ConvShape(B, 8, size, size // 2, 64, 7, 4, sy, 1, 3, 2, 1, 1, 3, 1)
        return _capi.load().tmq_ternary_conv2d_relu_maxpool_planar_f32_pays(planes, ctypes.byref(shape))
    assert [pays(1, 2, B) for B in (109, 110)] == [1, 0]
    for planes in (1, 2):
        assert [pays(planes, 1, B) for B in (54, 55)] == [1, 0]
    assert [pays(4, 1, B) for B in (36, 37)] == [1, 0]
    assert pays(3, 1, 1000) == 1 and all(pays(planes, 2, 1000) for planes in (2, 3, 4))
    assert pays(3, 2, 1, 0) == 0 and pays(5, 2, 1) == 0 and pays(0, 2, 1) == 0
