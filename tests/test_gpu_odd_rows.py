"""The two-kernel backward of contiguous 16-bit SAPA-B tensors whose rows have an odd number of cells."""
import pytest
import torch

import sapa_amd
from sapa_amd import _lib
from sapa_amd.sapa_func import _direct_serves
from test_gpu_fused16_range import exact_gradients, gradients, one_rounding, rel, same_non_finite

pytestmark = pytest.mark.gpu


def _operands(dtype, B, d, C, H, W):
    g = torch.Generator(device='cuda').manual_seed(H * W)
    shapes = ((B, d, 2 * H, 2 * W), (B, d, H, W), (B, C, H, W), (B, C, 2 * H, 2 * W))
    return [torch.randn(s, generator=g, device='cuda').mul(0.6).to(dtype) for s in shapes]


@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16])
@pytest.mark.parametrize('B,d,C,H,W', [
    (1, 16, 16, 4, 17),      # the smallest width served; rows end two children into a piece
    (2, 24, 40, 5, 19),      # ... six into one; ragged channel chunks, images of an odd number of cells
    (2, 17, 33, 3, 33),      # an odd number of channels too: the last dword of a tensor is half its own
    (1, 32, 64, 33, 31),     # one tile of cell blocks, its last one past the image
    (1, 40, 24, 3, 67),      # several tiles, fewer rows than a block
])
def test_gradients_of_odd_rows(dtype, B, d, C, H, W):
    """All gradients and one at a time against the fp64 operators.  Bar: one rounding of the result to its
    type leaves a relative error of eps / 2 / sqrt(3) at most; weight pairs and fp32 sums are far below."""
    *ops, go = _operands(dtype, B, d, C, H, W)
    assert _direct_serves(*ops, 5, 2, False)
    wide = [t.double().requires_grad_() for t in ops]
    want = torch.autograd.grad(sapa_amd.sapa_fused(*wide, 5, 2), wide, go.double())
    bar = torch.finfo(dtype).eps / 2 / 3 ** 0.5 * 1.2
    for needs in ((True, True, True), (True, False, False), (False, True, False), (False, False, True)):
        leaves = [t.clone().requires_grad_(n) for t, n in zip(ops, needs)]
        got = torch.autograd.grad(sapa_amd.sapa_fused(*leaves, 5, 2), [t for t in leaves if t.requires_grad], go)
        for a, b in zip(got, [w for w, n in zip(want, needs) if n]):
            rel = ((a.double() - b).norm() / b.norm()).item()
            assert rel <= bar and a.is_contiguous(), (needs, a.shape, rel)


def test_weights_hold_fp32s_precision():
    """Every cell in the window of one child with a query and a gradient: each of grad_value and grad_key is one weight
    times a bf16 number, rounded once.  fp32 arithmetic puts less than 2^-12 of them on the other side of a rounding
    (errors of 2^-20 at most, of a spacing of 2^-7 .. 2^-8); weights of 16 bits put more than 2^-11 there."""
    B, d, C, H, W = 16, 16, 16, 50, 85
    q, key, v, go = _operands(torch.bfloat16, B, d, C, H, W)
    child = torch.zeros(2 * H, 2 * W, dtype=torch.bool, device='cuda')
    child[4::10, 5::10] = True
    q, go = q * child, go * child
    wide = [t.double().requires_grad_() for t in (q, key, v)]
    want = torch.autograd.grad(sapa_amd.sapa_fused(*wide, 5, 2), wide, go.double())
    leaves = [t.clone().requires_grad_() for t in (q, key, v)]
    got = torch.autograd.grad(sapa_amd.sapa_fused(*leaves, 5, 2), leaves, go)
    for a, b in zip(got[1:], want[1:]):
        differ = (a != b.bfloat16()).double().mean().item()
        assert differ < 2.0 ** -12, differ


@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16])
@pytest.mark.parametrize('value', [float('nan'), float('inf')])
@pytest.mark.parametrize('which', [0, 1, 2, 3])
@pytest.mark.parametrize('C,H,W', [(40, 11, 23), (33, 9, 67)])
def test_non_finite_values_stay_where_they_belong(C, H, W, which, value, dtype):
    """Results that are stored half a dword over and formed again term by term behind it: at the ends of rows and
    images, one tile of cell blocks and several."""
    *ops, go = _operands(dtype, 2, 24, C, H, W)
    t = (*ops, go)[which]
    t[0, 3, 5, 0] = value
    t[1, 7, -1, -1] = value
    t[1, 2, 4, t.size(3) // 2] = -value
    assert _direct_serves(*ops, 5, 2, False)
    for got, want in zip(gradients(ops, go), exact_gradients(ops, go)[1:]):
        assert same_non_finite(got, want)
        ok = torch.isfinite(want)
        assert rel(got[ok], want[ok]) <= one_rounding(dtype)


def test_scratch_of_three_floats_per_pixel_does_not_serve_odd_rows():
    """The entry point whose scratch holds no padded copies refuses them and writes nothing."""
    q, key, v, go = _operands(torch.bfloat16, 1, 16, 16, 4, 17)
    scratch = torch.empty(3 * 8 * 34, dtype=torch.float32, device='cuda')
    grads = [torch.full_like(t, 7.0) for t in (q, key, v)]
    args = [_lib.ptr(t) for t in (go, q, key, v, scratch, *grads)]
    status = _lib.call_status('sapa_fused_backward_direct', q.device, *args, 1, 16, 16, 4, 17, 5, 2, 0,
                              _lib.dtype_code(q))
    assert status == _lib.UNSUPPORTED and all(bool((t == 7.0).all()) for t in grads)


@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16])
@pytest.mark.parametrize('B,C,H,W', [(16, 256, 43, 29), (8, 128, 51, 83), (4, 64, 51, 83), (16, 128, 43, 29)])
def test_training_output_of_odd_rows_as_with_kept_weights(dtype, B, C, H, W):
    """The output of a training step is, bit for bit, that of the one that keeps its fp32 weights, both where it is
    aggregated with them (the first two sizes) and where it comes from the one-launch forward."""
    q, key, v, _ = _operands(dtype, B, 32, C, H, W)
    leaves = [t.requires_grad_() for t in (q, key, v)]
    out = sapa_amd.sapa_fused(*leaves, 5, 2)
    kept = sapa_amd.sapa_fused(*leaves, 5, 2, save_attention=True)
    assert torch.equal(out, kept)
    assert not any(t.size(1) == 25 for t in out.grad_fn.saved_tensors)


def _behind(t, k):
    """t's values behind k others."""
    return torch.empty(t.numel() + k, dtype=t.dtype, device=t.device)[k:].copy_(t.reshape(-1)).view_as(t)


def test_tensors_that_begin_anywhere(monkeypatch):
    """Key, value and the output's gradient: the same gradients from the operands, also from the middle of a dword on.
    A query between two 16-byte pieces: the forward pass keeps the weights, and the backward pass chains over them."""
    q, key, v, go = _operands(torch.bfloat16, 2, 17, 33, 9, 33)
    names, call = [], _lib.call_status
    monkeypatch.setattr(_lib, 'call_status', lambda name, *a: names.append(name) or call(name, *a))

    def step(q, key, v, go):
        names.clear()
        leaves = [t.detach().requires_grad_() for t in (q, key, v)]
        out = sapa_amd.sapa_fused(*leaves, 5, 2)
        return (out,) + torch.autograd.grad(out, leaves, go), list(names)
    want, route = step(q, key, v, go)
    assert route == ['sapa_fused_backward_direct_ws']
    for k, at in ((1, 1), (1, 2), (1, 3), (4, 3)):
        ops = [q, key, v, go]
        ops[at] = _behind(ops[at], k)
        got, route = step(*ops)
        assert route == ['sapa_fused_backward_direct_ws']
        # (the output's low-res rows come through another kernel where they begin inside a dword)
        assert all(torch.equal(a, b) for a, b in zip(got[1:], want[1:]))
    got, route = step(_behind(q, 4), key, v, go)
    assert route == ['sapa_fused_forward_attn', 'sapa_fused_backward_attn']
    bar = torch.finfo(q.dtype).eps / 2 / 3 ** 0.5 * 1.2 * 2         # (one rounding of each)
    assert all(((a.double() - b.double()).norm() / b.double().norm()).item() <= bar for a, b in zip(got, want))
