"""The matrix-instruction kernels of 16-bit SAPA-B at the ends of their range: few channels, many
workgroups, large and small values, rows that end inside a 16-byte piece, non-finite values."""
import pytest
import torch

pytestmark = pytest.mark.gpu

ORDERS = {False: torch.contiguous_format, True: torch.channels_last}


def draw(g, shape, dtype, scale=1.0, channels_last=False):
    t = torch.randn(shape, generator=g, device='cuda') * scale
    return t.to(dtype).contiguous(memory_format=ORDERS[channels_last])


def exact_gradients(ops, go, K=5, s=2):
    """(output, gradients) of the operator in float64 on the same values"""
    import sapa_amd
    wide = [t.detach().double().contiguous().requires_grad_() for t in ops]
    out = sapa_amd.sapa_fused(*wide, K, s)
    return (out.detach(),) + torch.autograd.grad(out, wide, go.double().contiguous())


def gradients(ops, go, K=5, s=2):
    import sapa_amd
    leaves = [t.detach().clone(memory_format=torch.preserve_format).requires_grad_() for t in ops]
    return torch.autograd.grad(sapa_amd.sapa_fused(*leaves, K, s), leaves, go)


def rel(got, want):
    return ((got.double() - want).norm() / want.norm()).item()


def one_rounding(dtype):
    """relative error (2-norm) that one rounding of every result to `dtype` leaves at most, and a fifth"""
    return torch.finfo(dtype).eps / 2 / 3 ** 0.5 * 1.2


@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16])
@pytest.mark.parametrize('channels_last', [False, True])
@pytest.mark.parametrize('d', [8, 16])
def test_backward_of_one_chunk_of_keys(dtype, channels_last, d):
    """d of one staged chunk, several chunks of values, more workgroups than CUs: what the cell kernel
    reads right behind its first wait has to be there.  The same bits in every run."""
    g = torch.Generator(device='cuda').manual_seed(d)
    B, C, H, W = 16, 72, 64, 64
    shapes = ((B, d, 2 * H, 2 * W), (B, d, H, W), (B, C, H, W), (B, C, 2 * H, 2 * W))
    *ops, go = (draw(g, s, dtype, 0.6, channels_last) for s in shapes)
    first = gradients(ops, go)
    for got, want in zip(first, exact_gradients(ops, go)[1:]):
        assert rel(got, want) <= one_rounding(dtype)
    for _ in range(4):
        assert all(torch.equal(a, b) for a, b in zip(gradients(ops, go), first))


@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16])
@pytest.mark.parametrize('channels_last', [False, True])
@pytest.mark.parametrize('W', [18, 20, 22, 23])
def test_backward_with_logits_in_the_hundreds(dtype, channels_last, W):
    """Softmaxes that are almost one cell, and rows whose last 16-byte piece of children (W = 18, 22; of
    their statistics: W = 23) runs over into the next row: the products of those children with this
    row's cells are beyond what the exponential holds and must not count.  Bar: one rounding, and the fp32 logits' own error (64 * 2^-24 * 500 = 2e-3 at most, a
    tenth of that in the norm)."""
    g = torch.Generator(device='cuda').manual_seed(W)
    B, d, C, H = 2, 64, 24, 9
    q, k, v, go = ((B, d, 2 * H, 2 * W), (B, d, H, W), (B, C, H, W), (B, C, 2 * H, 2 * W))
    ops = [draw(g, q, dtype, 5.0, channels_last), draw(g, k, dtype, 5.0, channels_last), draw(g, v, dtype, 1.0, channels_last)]
    go = draw(g, go, dtype, 1.0, channels_last)
    want = exact_gradients(ops, go)[1:]
    for got, w in zip(gradients(ops, go), want):
        assert bool(torch.isfinite(got).all())
        assert rel(got, w) <= one_rounding(dtype) + 2e-4
