"""The fp32 training step on both sides of the number of tiles where its similarity stages change their geometry."""
import pytest
import torch

import sapa_amd

pytestmark = pytest.mark.gpu


# (an image alone has 42 / 36 / 1 tiles of 16 x 8 parents; the batches 504, 546, 540 and 2: up to 512 take those tiles;
# rows of whole and of no whole vectors, one cell over a tile)
@pytest.mark.parametrize('B,d,C,H,W', [(12, 16, 24, 50, 84), (13, 16, 24, 50, 84), (15, 8, 9, 65, 49), (2, 5, 3, 7, 3)])
def test_batch_and_single_images_agree(B, d, C, H, W):
    """The same terms in the same order whichever tiles compute them: every bit equal."""
    g = torch.Generator(device='cuda').manual_seed(H)
    draw = lambda *s: torch.randn(*s, generator=g, device='cuda')
    q, k, v, go = draw(B, d, 2 * H, 2 * W), draw(B, d, H, W), draw(B, C, H, W), draw(B, C, 2 * H, 2 * W)

    def step(*t):
        leaves = [x.clone().requires_grad_() for x in t[:3]]
        out = sapa_amd.sapa_fused(*leaves, 5, 2)
        return (out.detach(),) + torch.autograd.grad(out, leaves, t[3])
    full = step(q, k, v, go)
    for n in (0, B - 1):
        one = step(*(t[n:n + 1] for t in (q, k, v, go)))
        for name, a, b in zip(('out', 'grad_query', 'grad_key', 'grad_value'), full, one):
            assert torch.equal(a[n:n + 1], b), (name, n)
