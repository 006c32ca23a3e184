"""Low-res gradients whose channels are split over workgroups in slices that do not divide them."""
import pytest
import torch

import sapa_amd

pytestmark = pytest.mark.gpu


# (slices of 8 channels, the last of 5; of 16, the last of 2; of 20, the last of 13; a single channel; tiles of 12 and
# of 15 waves, two each, ragged in x and y)
@pytest.mark.parametrize('B,C,H,W', [(1, 37, 21, 70), (8, 130, 29, 47), (16, 33, 50, 84), (1, 1, 24, 50), (11, 15, 39, 79),
                                     (11, 62, 19, 47), (11, 37, 51, 53), (8, 37, 50, 82)])
@pytest.mark.parametrize('dtype', [torch.float32, torch.bfloat16])
def test_every_channel_of_every_slice(dtype, B, C, H, W):
    """Integers: every product and sum is exact in fp32, in any order (the result rounded once to 16 bits)."""
    g = torch.Generator(device='cuda').manual_seed(C)
    draw = lambda *shape: torch.randint(-3, 4, shape, generator=g, device='cuda').to(dtype)
    attn, grad = draw(B, 25, 2 * H, 2 * W), draw(B, C, 2 * H, 2 * W)
    value = torch.zeros(B, C, H, W, dtype=dtype, device='cuda').requires_grad_()
    sapa_amd.av(attn, value, 5, 2).backward(grad)
    a, o = attn.double().view(B, 25, 1, H, 2, W, 2), grad.double().view(B, C, H, 2, W, 2)
    padded = torch.zeros(B, C, H + 4, W + 4, dtype=torch.float64, device='cuda')
    for k in range(25):
        padded[:, :, k // 5:k // 5 + H, k % 5:k % 5 + W] += (a[:, k] * o).sum((3, 5))
    assert torch.equal(value.grad, padded[:, :, 2:-2, 2:-2].to(dtype))
