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


# (eight waves on channels-last features: runs of 2 tiles of each of 8 waves, and of 3 tiles of 7 waves, a ragged last tile
# in both; weights shared by the images: 7 of 8 waves; 12 waves and a last block of 8 outputs; planes of no whole lines;
# planes of whole lines, runs of 2 tiles of 7 waves)
@pytest.mark.parametrize('B,C,O,H,W', [(16, 128, 32, 50, 84), (9, 128, 32, 100, 169), (2, 512, 72, 100, 168), (2, 256, 264, 100, 168),
                                       (3, 64, 40, 150, 134), (8, 64, 160, 64, 64)])
def test_runs_of_tiles_and_shared_weights(B, C, O, H, W):
    """As above; weights shared by the images through project_shared."""
    if O == 32:
        g = torch.Generator(device='cuda').manual_seed(H)
        x = torch.randn(B, C, H, W, generator=g, device='cuda')
        w = torch.randn(B, O, C, generator=g, device='cuda') * 0.1
        got = _lib.project_nhwc(x.contiguous(memory_format=torch.channels_last), w)
        results, weights = [got.reshape(B, O, H * W)], w
    else:
        g = torch.Generator(device='cuda').manual_seed(W)
        x = torch.randn(B, C, H, W, generator=g, device='cuda')
        w = torch.randn(O, C, generator=g, device='cuda') * 0.1
        results = [_lib.project_shared(t, w, None, cl).reshape(B, O, H * W)
                   for t, cl in ((x, False), (x, True), (x.contiguous(memory_format=torch.channels_last), True))]
        weights = w.expand(B, O, C)
    for b in range(B):
        wide = x[b].double().view(C, H * W)
        want, bar = weights[b].double() @ wide, (weights[b].double().abs() @ wide.abs()) * 2.0 ** -21
        for r in results:
            assert bool(((r[b].double() - want).abs() <= bar).all()), b
