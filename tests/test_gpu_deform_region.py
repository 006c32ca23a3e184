"""The one-kernel backward of fused SAPA-D for 16-bit tensors at up_factor 2: strips of parent rows in one and in many
steps round the window ring, ragged edges, far points, values that are not finite."""
import pytest
import torch

import sapa_amd
from helpers import deform_fused_backward_oracle, gen, randn
from test_gpu_sapa_d import DEV, dev, make

pytestmark = pytest.mark.gpu
NAMES = ('grad_query', 'grad_key', 'grad_value', 'grad_offset')
# B, G, dq, cg, H, W, P, offset scale: so few strips are split into segments of one row each (one step);
# a ragged strip beside a whole one; rows of two pixels over a multiple of 4; one narrow strip; far points in both
# lane mappings
SHAPES = [(1, 2, 32, 64, 37, 21, 25, 0.75), (2, 1, 24, 40, 20, 9, 16, 2.0), (1, 1, 8, 8, 50, 3, 2, 0.7),
          (1, 2, 32, 64, 17, 13, 32, 6.0), (3, 2, 16, 24, 3, 5, 9, 1.0), (1, 1, 32, 48, 33, 16, 17, 1.5)]


def _inputs(shape, dtype, seed=400):
    B, G, dq, cg, H, W, P, oscale = shape
    g = gen(seed)
    q, key, v, off, _ = make(g, (B, G, dq, cg, H, W, P, 2), off_scale=oscale)
    off = off.floor() + (off - off.floor()).clamp(0.2, 0.8)      # rounding must not cross a cell's edge
    go = randn(g, B, G * cg, 2 * H, 2 * W)
    return [t.to(dtype) for t in (q, key, v, off, go)]


def _gradients(q, key, v, off, go, P, G):
    t = [x.requires_grad_() for x in dev(q, key, v, off)]
    out = sapa_amd.deform_sapa_fused(*t, P, 2, G)
    return torch.autograd.grad(out, t, go.to(DEV))


@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16])
@pytest.mark.parametrize('shape', SHAPES, ids=['-'.join(map(str, s)) for s in SHAPES])
def test_against_the_exact_chain(coracle, shape, dtype):
    """One rounding of each gradient (half a spacing: 2^-8 / 2^-11 of the value at most), and the fp32 chain's
    own errors, of some 1e-5 of what cancels in it (up to 40 rms over these sizes)."""
    P, G = shape[6], shape[1]
    q, key, v, off, go = _inputs(shape, dtype)
    want = deform_fused_backward_oracle(coracle, go.float(), q.float(), key.float(), v.float(), off.float(), P, 2, G)
    rel = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    for got, w, name in zip(_gradients(q, key, v, off, go, P, G), want, NAMES):
        err, rms = (got.cpu().double() - w).abs(), w.pow(2).mean().sqrt()
        worst = (err / (rel * w.abs() + 4e-4 * rms)).max().item()
        assert worst <= 1, f'{name}: {worst}'


def _steps(B, G, H, W):
    """Rows of parents per workgroup: the launcher's rule (the shortest of rounds of 256 workgroups times rows + 4)."""
    columns, best = (W + 7) // 8 * G * B, None
    for k in range(1, H + 1):
        if k > 1 and columns * (k - 1) >= 4 * 256:
            break
        rows = -(-H // k)
        time = -(-(columns * -(-H // rows)) // 256) * (rows + 4)
        if best is None or time < best[0]:
            best = time, rows
    return best[1]


# 256 strips, whole: 37 steps go round the ring of 15 window rows twice and more; a strip of 8 parents and a ragged one,
# rows of 26 pixels; both lane mappings, samples far from their parents and near
MANY = [(32, 4, 8, 8, 37, 13, 9, 0.9), (32, 4, 24, 40, 37, 13, 25, 2.5), (64, 2, 32, 64, 33, 9, 16, 0.75)]


@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16])
@pytest.mark.parametrize('shape', MANY, ids=['-'.join(map(str, s)) for s in MANY])
def test_many_steps(coracle, shape, dtype):
    """As above, the first and the last image."""
    B, G, dq, cg, H, W, P, _ = shape
    assert _steps(B, G, H, W) > 2 * 15
    ops = _inputs(shape, dtype, seed=406)
    got = _gradients(*ops, P, G)
    rel = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    for n in (0, B - 1):
        q, key, v, off, go = (t[n:n + 1].float() for t in ops)
        want = deform_fused_backward_oracle(coracle, go, q, key, v, off, P, 2, G)
        for a, w, name in zip(got, want, NAMES):
            err, rms = (a[n:n + 1].cpu().double() - w).abs(), w.pow(2).mean().sqrt()
            worst = (err / (rel * w.abs() + 4e-4 * rms)).max().item()
            assert worst <= 1, f'{name} of image {n}: {worst}'


@pytest.mark.parametrize('which', ['query', 'key', 'value', 'grad_out'])
@pytest.mark.parametrize('row', [2, 31])
def test_non_finite_values_in_one_of_many_steps(coracle, which, row):
    """A value that is not finite in an early or late step: its image's gradients are not finite where the exact chain's are
    not, and right elsewhere; its neighbour in the batch has none."""
    shape = (32, 4, 8, 8, 37, 13, 9, 0.9)
    ops = dict(zip(('query', 'key', 'value', 'offset', 'grad_out'), _inputs(shape, torch.float16, seed=407)))
    t = ops[which]
    t[5, 3, row * t.size(2) // 37 + 1, 5] = float('inf')
    got = _gradients(*ops.values(), 9, 4)
    for n in (5, 6):
        q, key, v, off, go = (x[n:n + 1].float() for x in ops.values())
        want = deform_fused_backward_oracle(coracle, go, q, key, v, off, 9, 2, 4)
        for a, w, name in zip(got, want, NAMES):
            a, fine = a[n:n + 1].cpu().double(), torch.isfinite(w)
            assert torch.equal(torch.isfinite(a), fine), (name, n)
            err, rms = (a - w)[fine].abs(), w[fine].pow(2).mean().sqrt()
            assert bool((err <= 2.0 ** -11 * w[fine].abs() + 4e-4 * rms).all()), (name, n)


@pytest.mark.parametrize('which', ['query', 'key', 'value', 'grad_out'])
@pytest.mark.parametrize('bad', [float('inf'), float('nan')])
def test_non_finite_values_reach_what_they_belong_to(coracle, which, bad):
    """Gradients that the exact chain has as infinite or NaN, and no others, are not finite."""
    shape = (1, 2, 16, 24, 19, 11, 9, 0.7)
    q, key, v, off, go = _inputs(shape, torch.bfloat16, seed=401)
    t = {'query': q, 'key': key, 'value': v, 'grad_out': go}[which]
    t[0, 3, 6, 5] = bad
    t[0, t.size(1) - 1, 12, 9] = bad
    want = deform_fused_backward_oracle(coracle, go.float(), q.float(), key.float(), v.float(), off.float(), 9, 2, 2)
    for got, w, name in zip(_gradients(q, key, v, off, go, 9, 2), want, NAMES):
        assert torch.equal(torch.isfinite(got).cpu(), torch.isfinite(w)), name


def test_gradients_of_any_size_in_fp16(coracle):
    """fp16 gradients that are small or large as a whole (loss scales), and pixels 2^-12 apart."""
    shape = (1, 1, 32, 64, 18, 17, 25, 0.75)
    q, key, v, off, go = _inputs(shape, torch.float32, seed=402)
    go[..., ::2] *= 2.0 ** -12
    for scale in (2.0 ** -10, 2.0 ** 6):
        a = [t.half() for t in (q, key, v, off, go * scale)]
        want = deform_fused_backward_oracle(coracle, a[4].float(), *(t.float() for t in a[:4]), 25, 2, 1)
        for got, w, name in zip(_gradients(*a, 25, 1), want, NAMES):
            err, rms = (got.cpu().double() - w).abs(), w.pow(2).mean().sqrt()
            # (2^-25: half the smallest spacing of the type)
            assert bool((err <= 2.0 ** -11 * w.abs() + 4e-4 * rms + 2.0 ** -25).all()), (name, scale)


@pytest.mark.parametrize('which', ['grad_out', 'key'])
@pytest.mark.parametrize('big', [2.0 ** 98, 2.0 ** -98])
def test_bf16_operands_near_the_types_ends(coracle, which, big):
    """bf16 values of some 2^98 or 2^-98, whose gradients fp32 holds: the same as of ordinary ones but for the scale."""
    shape = (1, 1, 32, 64, 18, 17, 25, 0.75)
    q, key, v, off, go = _inputs(shape, torch.bfloat16, seed=403)
    want = deform_fused_backward_oracle(coracle, go.float(), q.float(), key.float(), v.float(), off.float(), 25, 2, 1)
    if which == 'grad_out':
        got, scale = _gradients(q, key, v, off, go * big, 25, 1), (big, big, big, big)
    else:
        got, scale = _gradients(q / big, key * big, v, off, go, 25, 1), (big, 1 / big, 1.0, 1.0)
    for a, w, f, name in zip(got, want, scale, NAMES):
        err, rms = (a.cpu().double() / f - w).abs(), w.pow(2).mean().sqrt()
        assert bool((err <= 2.0 ** -8 * w.abs() + 4e-4 * rms).all()), name


def test_corner_weights_hold_24_bits_in_fp16():
    """Cells that one sample of one pixel reaches, with a gradient of the output of 1: grad_value is the corner's weight,
    rounded once.  Equal logits of 3 points, two of them outside the image: weights of fl(1/3) times a corner's
    share, in fixed point of 2^-30 (half a million of them: some would round the other way with a bit less)."""
    B, G, H, W, P = 16, 8, 64, 64, 3
    g = torch.Generator(device='cuda').manual_seed(404)
    q = torch.zeros(B, 8 * G, 2 * H, 2 * W, device='cuda')
    key, v = (torch.randn(B, 8 * G, H, W, generator=g, device='cuda') for _ in range(2))
    off = torch.full((B, G, P, 2, 2 * H, 2 * W), 1000.0, device='cuda')
    # (x, y) of every second parent, of all sizes below 1
    steps = torch.exp2(-4 * torch.rand(B, G, 2, 32, 32, generator=g, device='cuda') - 0.1).half().float()
    off[:, :, 0, :, ::4, ::4] = steps
    go = torch.zeros_like(q)
    go[..., ::4, ::4] = 1
    at = 2.0 * torch.arange(32, device='cuda')
    kw, kh = steps[:, :, 0] + at, steps[:, :, 1] + at[:, None]
    low_w, low_h = kw.floor(), kh.floor()
    lw, lh = kw - low_w, kh - low_h
    want = torch.zeros(B, G, H + 1, W + 1, device='cuda')
    n, grp = (torch.arange(k, device='cuda').view(s) for k, s in ((B, (B, 1, 1, 1)), (G, (1, G, 1, 1))))
    third = torch.tensor(1.0, device='cuda') / 3 * 2.0 ** 30
    for dy, dx, share in ((0, 0, (1 - lh) * (1 - lw)), (0, 1, (1 - lh) * lw), (1, 0, lh * (1 - lw)), (1, 1, lh * lw)):
        want[n, grp, low_h.long() + dy, low_w.long() + dx] = (third * share).round() * 2.0 ** -30
    want = want[:, :, :H, :W].half().unsqueeze(2).expand(B, G, 8, H, W).reshape(B, 8 * G, H, W)
    t = [x.half().requires_grad_() for x in (q, key, v, off.view(B, 2 * G * P, 2 * H, 2 * W))]
    got = torch.autograd.grad(sapa_amd.deform_sapa_fused(*t, P, 2, G), t, go.half())
    assert torch.equal(got[2], want)


@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16])
@pytest.mark.parametrize('shape', [(1, 1, 24, 40, 20, 9, 16, 1.0), (2, 2, 32, 64, 7, 21, 9, 1.0)], ids=['18-wide', '42-wide'])
def test_last_pixels_of_rows_that_end_inside_a_piece(shape, dtype):
    """Rows of 4 n + 2 pixels, the tensors' last ones with NaN right behind them: the piece that runs over the end brings
    the two pixels in front of it and nothing that counts."""
    P, G = shape[6], shape[1]
    plain = [t.to(DEV) for t in _inputs(shape, dtype, seed=405)]

    def before_nan(t):
        room = torch.full((t.numel() + 64,), float('nan'), dtype=dtype, device=DEV)
        return room[:t.numel()].copy_(t.detach().reshape(-1)).view_as(t)
    want = _gradients(*plain, P, G)
    got = _gradients(*(before_nan(t) for t in plain), P, G)
    assert torch.equal(got[0], want[0]) and torch.equal(got[3], want[3])
    for a, b in zip(got[1:3], want[1:3]):           # (atomic sums, in any order)
        torch.testing.assert_close(a, b, rtol=torch.finfo(dtype).eps, atol=1e-5)
    for t, grads in ((plain[0], got[0]), (plain[3], got[3])):
        assert bool(torch.isfinite(grads).all()) and grads[..., -1, -2:].abs().max() > 0
