"""Fused SAPA-D of contiguous fp32 tensors with up to 9 points (samples gathered from an LDS window, points in registers)."""
import pytest
import torch

import sapa_amd
from helpers import assert_f32_close, gen, randn
from sapa_amd import _lib

pytestmark = pytest.mark.gpu

# B, G, dq, cg, H, W, P, offset scale: whole tiles of 8 x 16 parents; ragged ones, chunks of 16 channels that are not
# full, one more than a chunk, fewer points than registers, every sample beyond the window or the image, the narrowest image
SHAPES = [(1, 4, 32, 64, 16, 16, 9, 0.75), (2, 2, 10, 20, 9, 17, 5, 1.5), (1, 3, 17, 33, 7, 31, 6, 6.0),
          (2, 1, 5, 7, 13, 9, 1, 3.0), (1, 1, 16, 16, 24, 24, 8, 40.0)]


@pytest.mark.parametrize('shape', SHAPES, ids=['-'.join(map(str, s)) for s in SHAPES])
def test_against_the_oracle(coracle, shape):
    B, G, dq, cg, H, W, P, scale = shape
    g = gen(71)
    q, key, v = randn(g, B, G * dq, 2 * H, 2 * W), randn(g, B, G * dq, H, W), randn(g, B, G * cg, H, W)
    off = randn(g, B, 2 * G * P, 2 * H, 2 * W) * scale
    got = sapa_amd.deform_sapa_fused(*(t.cuda() for t in (q, key, v, off)), P, 2, G).cpu()
    assert _lib.lib().sapa_hip_last_kernel() == b'deform_gather_kernel'
    assert_f32_close(got, coracle.deform_sapa_fused(q, key, v, off, P, 2, G, 'f32'), 'deform fused')


def test_values_that_are_not_finite_stay_where_they_are_sampled(coracle):
    """Infinite queries meet samples outside the image (logit 0), infinite values only the samples that touch them."""
    G, P, H, W = 2, 7, 11, 18
    g = gen(72)
    q, key, v = randn(g, 1, G * 6, 2 * H, 2 * W), randn(g, 1, G * 6, H, W), randn(g, 1, G * 20, H, W)
    off = randn(g, 1, 2 * G * P, 2 * H, 2 * W) * 3
    q[0, 1, 5, 7] = float('inf')
    v[0, 3, 6, 9] = float('inf')
    key[0, 2, 4, 4] = float('nan')
    off[0, :, 0, 0] = -30.                       # every sample of a pixel with an infinite query outside
    q[0, :, 0, 0] = float('inf')
    off[0, 1, 3, 3], off[0, 2, 3, 3] = float('nan'), float('inf')
    got = sapa_amd.deform_sapa_fused(*(t.cuda() for t in (q, key, v, off)), P, 2, G).cpu()
    want = coracle.deform_sapa_fused(q, key, v, off, P, 2, G, 'f32')
    assert torch.equal(torch.isfinite(got), torch.isfinite(want)) and torch.equal(got.isnan(), want.isnan())
    assert torch.equal(got[0, :, 0, 0], torch.zeros(G * 20))
    ok = torch.isfinite(want)
    assert_f32_close(got[ok], want[ok], 'finite outputs')


# slices of one chunk each; 100 tiles: of three chunks and two, of two and one that is partial
@pytest.mark.parametrize('B,G,cg,H,W,scale', [(33, 2, 20, 16, 16, 0.75), (33, 2, 33, 16, 16, 6.0), (33, 2, 64, 16, 16, 3.0),
                                              (33, 2, 100, 16, 16, 1.5), (3, 4, 80, 40, 80, 0.75), (3, 4, 44, 40, 80, 3.0)])
def test_value_channels_in_slices(B, G, cg, H, W, scale):
    """An image by itself, its value channels in up to a slice per 16, gives what it gives in a batch whose tiles take all
    of them: whole chunks, a last one partial, samples beyond the window."""
    P = 7
    g = gen(73)
    q, key, v = randn(g, B, G * 20, 2 * H, 2 * W), randn(g, B, G * 20, H, W), randn(g, B, G * cg, H, W)
    off = randn(g, B, 2 * G * P, 2 * H, 2 * W) * scale
    q, key, v, off = (t.cuda() for t in (q, key, v, off))
    got = sapa_amd.deform_sapa_fused(q, key, v, off, P, 2, G)
    for n in (0, B // 2, B - 1):
        i = slice(n, n + 1)
        assert torch.equal(got[i], sapa_amd.deform_sapa_fused(*(t[i].contiguous() for t in (q, key, v, off)), P, 2, G))
        assert _lib.lib().sapa_hip_last_kernel() == b'deform_gather_kernel'


@pytest.mark.parametrize('P', [2, 4, 8])
@pytest.mark.parametrize('scale', [3.0, 6.0])
def test_samples_beyond_the_window_are_added_in_the_order_of_the_points(coracle, P, scale):
    """Equal logits make every weight exactly 1 / P: the output is deform_av's, in its order of sums, bit for bit,
    also where samples lie in the image but not in the tile's window."""
    G, cg, H, W = 2, 37, 33, 40
    g = gen(74)
    q, key = torch.zeros(1, G * 3, 2 * H, 2 * W), randn(g, 1, G * 3, H, W)
    v, off = randn(g, 1, G * cg, H, W), randn(g, 1, 2 * G * P, 2 * H, 2 * W) * scale
    got = sapa_amd.deform_sapa_fused(*(t.cuda() for t in (q, key, v, off)), P, 2, G, matrix_form=False).cpu()
    assert _lib.lib().sapa_hip_last_kernel() == b'deform_gather_kernel'
    attn = torch.full((1, G, P, 2 * H, 2 * W), 1. / P)
    assert torch.equal(got, coracle.deform_av(attn, v, off, P, 2, G, 'f32'))
