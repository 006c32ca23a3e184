"""The fp32 projection where its workgroups take several tiles of 32 pixels per wave."""
import pytest
import torch

from sapa_amd import _lib

pytestmark = pytest.mark.gpu


# (one round: 2 tiles per wave and 7 of 12 waves; 3 and 11 with a ragged last tile; two rounds of 6 tiles,
# the last wave's beyond the image)
@pytest.mark.parametrize('B,C,O,H,W', [(16, 64, 64, 49, 128), (16, 256, 64, 100, 168), (16, 512, 32, 97, 164),
                                       (128, 64, 32, 90, 86)])
def test_every_tile_of_every_wave(B, C, O, H, W):
    """Against float64 products.  Bar: the six largest of nine piece products and fp32 sums leave an error
    below 2^-21 of the sum of magnitudes."""
    g = torch.Generator(device='cuda').manual_seed(H)
    x = torch.randn(B, C, H, W, generator=g, device='cuda')
    w = torch.randn(B, O, C, generator=g, device='cuda') * 0.1
    planes = _lib.project_nchw(x, w)
    records = _lib.project_nhwc(x.contiguous(memory_format=torch.channels_last), w)
    for b in range(B):
        want = w[b].double() @ x[b].double().view(C, H * W)
        bar = (w[b].double().abs() @ x[b].double().abs().view(C, H * W)) * 2.0 ** -21
        assert bool(((planes[b].double().view(O, H * W) - want).abs() <= bar).all()), b
        assert torch.equal(records[b].reshape(O, H * W), planes[b].view(O, H * W)), b


# (8 and 12 waves per workgroup on both sides of where one takes over: tiles for exactly 8 waves of 256 workgroups
# and a few more, 256 -> 64 with 6 and 7 waves at work, two tiles for each of 8 waves; ragged last tiles)
@pytest.mark.parametrize('B,C,O,H,W', [(2, 256, 32, 256, 128), (2, 256, 32, 256, 130), (2, 64, 32, 300, 170), (3, 128, 32, 50, 86),
                                       (1, 256, 64, 224, 220), (1, 256, 64, 224, 212), (4, 512, 32, 256, 128), (1, 512, 32, 3, 4)])
def test_both_numbers_of_waves(B, C, O, H, W):
    test_every_tile_of_every_wave(B, C, O, H, W)
