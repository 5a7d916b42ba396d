"""The reordering conversion reduces the scan's partial maxima itself: whichever of them holds the largest value, at the
edges of the runs of 256 that its threads read and at the full 1024, the prescale is the one of the whole tensor."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("partials", [1, 2, 255, 256, 257, 511, 1024, 1500])
def test_every_partial_maximum_counts(cuda, partials):
    from tmq_amd import ops
    B, C, P = 1, 16, 256                        # 4096 values: what a workgroup of the scan takes per round
    x = torch.rand((B * partials, C, 16, P // 16), device=cuda) + 0.5
    flat = x.view(-1)
    for at in {0, flat.numel() - 1, flat.numel() // 2, min(255, partials - 1) * 4096, min(256, partials - 1) * 4096 + 4095}:
        kept = flat[at].clone()
        flat[at] = -7e8                         # s = 2^(11 - 30)
        hi, adjusted = ops.f32_to_f16_prescaled(x, None, 8, channels_last=True)
        assert torch.equal(adjusted, torch.full_like(adjusted, 2.0 ** 19))
        assert torch.equal(hi, (x * 2.0 ** -19).half())
        flat[at] = kept
