"""Kernels and dispatch branches at the sizes where they can go wrong: edges of tiles, remainders,
the first and last sizes of a range."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('channels_last_out', [False, True])
@pytest.mark.parametrize('dtype,C,O', [(torch.bfloat16, 256, 64), (torch.float16, 64, 32), (torch.float32, 128, 64)])
def test_projection_of_planes_with_two_workgroups_per_cu(dtype, C, O, channels_last_out):
    """More workgroups than CUs, so that result stores wait behind another workgroup's: every
    result against fp32 products of the same operands, four runs."""
    from sapa_amd import _lib
    g = torch.Generator(device='cuda').manual_seed(0)
    B, H, W = 2, 384, 384
    x = torch.randn(B, C, H, W, generator=g, device='cuda').to(dtype)
    w = (torch.randn(B, O, C, generator=g, device='cuda') * 0.05).to(dtype)
    b = torch.randn(B, O, generator=g, device='cuda').to(dtype)
    want = torch.bmm(w.float(), x.float().reshape(B, C, H * W)).view(B, O, H, W) + b.float()[:, :, None, None]
    # one rounding of the result to its type, fp32 sums of C products
    eps = torch.finfo(dtype).eps if dtype != torch.float32 else 0.0
    bar = 0.5 * eps * want.abs() + 2e-5
    for _ in range(4):
        got = _lib.project_nchw(x, w, b, channels_last_out=channels_last_out).float()
        assert int(((got - want).abs() > bar).sum()) == 0


def _rel(got, want):
    return ((got.double() - want).norm() / want.norm()).item()


@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16])
@pytest.mark.parametrize('channels_last,B,d,C,H,W', [
    (False, 1, 16, 16, 4, 16),      # the smallest width served
    (False, 2, 24, 40, 5, 18),      # ragged channel chunks, rows of 4 k + 2 cells, a last row of blocks of one row
    (False, 1, 32, 64, 33, 30),     # one tile of cell blocks, its last one past the image
    (False, 1, 40, 24, 3, 66),      # several tiles, fewer rows than a block
    (True, 1, 8, 8, 1, 3),          # the smallest tensors served
    (True, 2, 72, 40, 9, 17),       # ragged channel chunks, odd extents
    (True, 1, 64, 136, 15, 62),     # whole and partial tiles in both directions
])
def test_fused_backward_from_operands(dtype, channels_last, B, d, C, H, W):
    """The two-kernel backward of 16-bit tensors (sapa_fused_backward_direct) against the fp64
    operators, all gradients and one at a time.  Bar: one rounding of the result to its type leaves a
    relative error of eps / 2 / sqrt(3) at most; the 16-bit weight pairs and fp32 sums are far below."""
    import sapa_amd
    from sapa_amd.sapa_func import _direct_serves
    g = torch.Generator(device='cuda').manual_seed(H * W)
    shapes = ((B, d, 2 * H, 2 * W), (B, d, H, W), (B, C, H, W), (B, C, 2 * H, 2 * W))
    fmt = torch.channels_last if channels_last else torch.contiguous_format
    *ops, go = (torch.randn(s, generator=g, device='cuda').mul(0.6).to(dtype).contiguous(memory_format=fmt) for s in shapes)
    assert _direct_serves(*ops, 5, 2, channels_last)
    wide = [t.double().contiguous().requires_grad_() for t in ops]
    want = torch.autograd.grad(sapa_amd.sapa_fused(*wide, 5, 2), wide, go.double().contiguous())
    bar = torch.finfo(dtype).eps / 2 / 3 ** 0.5 * 1.2
    for needs in ((True, True, True), (True, False, False), (False, True, False), (False, False, True)):
        leaves = [t.clone(memory_format=torch.preserve_format).requires_grad_(n) for t, n in zip(ops, needs)]
        got = torch.autograd.grad(sapa_amd.sapa_fused(*leaves, 5, 2), [t for t in leaves if t.requires_grad], go)
        for a, b in zip(got, [w for w, n in zip(want, needs) if n]):
            assert _rel(a, b) <= bar and a.is_contiguous(memory_format=fmt), (needs, a.shape)


@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16])
@pytest.mark.parametrize('B,d,C,H,W', [
    (1, 16, 16, 4, 4),       # one block; the value channels cannot be split
    (2, 24, 40, 5, 7),       # odd rows inside one tile, ragged channel chunks
    (1, 17, 33, 3, 33),      # an odd number of channels and cells: the last dword of a tensor is half its own
    (3, 32, 256, 9, 18),     # value channels split over workgroups
    (2, 17, 33, 3, 33),      # images of an odd number of elements: the second starts in the middle of a dword
    (2, 32, 72, 21, 67),     # three tiles of an odd row
])
def test_fused_dense_window_kernel_edges(dtype, B, d, C, H, W):
    """The contiguous 16-bit dense-window forward where rows are odd or short and where its value
    channels are split, against the fp64 operator; bar as above."""
    import sapa_amd
    from sapa_amd import _lib
    g = torch.Generator(device='cuda').manual_seed(W)
    shapes = ((B, d, 2 * H, 2 * W), (B, d, H, W), (B, C, H, W))
    ops = [torch.randn(s, generator=g, device='cuda').mul(0.6).to(dtype) for s in shapes]
    with torch.no_grad():
        got = sapa_amd.sapa_fused(*ops, 5, 2)
        assert _lib.last_kernel() == 'sapa_b_wmat16_kernel'
        want = sapa_amd.sapa_fused(*[t.double() for t in ops], 5, 2)
    assert _rel(got, want) <= torch.finfo(dtype).eps / 2 / 3 ** 0.5 * 1.2


@pytest.mark.parametrize('dtype', [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize('in_cl,out_cl', [(False, False), (False, True), (True, True)])
@pytest.mark.parametrize('B,C,O,H,W', [
    (1, 64, 8, 2, 4),        # a part of one block of outputs, a part of one tile of pixels
    (2, 128, 72, 7, 8),      # one block and a remainder of 8
    (3, 256, 288, 9, 40),    # several blocks, the last one half full
    (1, 512, 40, 12, 34),    # blocks of 32 outputs
    (16, 256, 128, 16, 16),  # more workgroups than CUs for the 16-bit kernels
])
def test_projection_with_shared_weights(dtype, in_cl, out_cl, B, C, O, H, W):
    """sapa_project_shared against fp64 products of the same operands: fp32 within an error bound of
    a C-term fp32 dot product (C + 8 roundings of 2^-24 of the sum of magnitudes), 16-bit results one
    rounding further."""
    from sapa_amd import _lib
    g = torch.Generator(device='cuda').manual_seed(O)
    x = torch.randn(B, C, H, W, generator=g, device='cuda').to(dtype)
    if in_cl:
        x = x.contiguous(memory_format=torch.channels_last)
    w = torch.randn(O, C, 1, 1, generator=g, device='cuda').mul(0.05).to(dtype)
    b = torch.randn(O, generator=g, device='cuda').to(dtype)
    x64, w64 = x.double().contiguous().reshape(B, C, H * W), w.double().reshape(1, O, C).expand(B, O, C).contiguous()
    for bias in (b, None):
        got = _lib.project_shared(x, w, bias, channels_last_out=out_cl)
        assert got.is_contiguous(memory_format=torch.channels_last if out_cl else torch.contiguous_format)
        want = torch.bmm(w64, x64).view(B, O, H, W)
        mag = torch.bmm(w64.abs(), x64.abs()).view(B, O, H, W)
        if bias is not None:
            want, mag = want + b.double().view(1, O, 1, 1), mag + b.double().abs().view(1, O, 1, 1)
        bar = (C + 8) * 2.0 ** -24 * mag + (0.0 if dtype == torch.float32 else 0.5 * torch.finfo(dtype).eps * want.abs() + 1e-7)
        assert int(((got.double() - want).abs() > bar).sum()) == 0


@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16])
@pytest.mark.parametrize('K,s', [(7, 4), (5, 4), (3, 2)])
@pytest.mark.parametrize('B,d,C,H,W', [
    (1, 16, 16, 1, 4),       # one row, the smallest width
    (2, 24, 40, 5, 7),       # odd rows inside one tile, ragged channel chunks
    (2, 17, 33, 3, 21),      # an odd number of channels and cells: images start in the middle of a dword
    (3, 32, 136, 9, 18),     # several tiles of s = 4, a partial one; value channels split over workgroups
    (1, 32, 72, 6, 67),      # tiles of an odd row
    (16, 40, 64, 33, 64),    # more tiles than CUs
])
def test_fused_dense_window_kernel_other_windows(dtype, K, s, B, d, C, H, W):
    """The dense-window forward with a window piece per block, against the fp64 operator; bar as above."""
    import sapa_amd
    from sapa_amd import _lib
    g = torch.Generator(device='cuda').manual_seed(W)
    shapes = ((B, d, s * H, s * W), (B, d, H, W), (B, C, H, W))
    ops = [torch.randn(sh, generator=g, device='cuda').mul(0.6).to(dtype) for sh in shapes]
    with torch.no_grad():
        got = sapa_amd.sapa_fused(*ops, K, s)
        assert _lib.last_kernel() == 'sapa_b_wmat16_kernel'
        want = sapa_amd.sapa_fused(*[t.double() for t in ops], K, s)
    assert _rel(got, want) <= torch.finfo(dtype).eps / 2 / 3 ** 0.5 * 1.2


@pytest.mark.parametrize('dtype', [torch.float32, torch.bfloat16])
@pytest.mark.parametrize('B,d,C,H,W', [
    (1, 32, 64, 32, 32),      # one image
    (3, 17, 5, 7, 19),        # ragged tiles, channels that fill no chunk
    (1, 40, 256, 64, 64),     # the last size of the aggregation on this kernel
    (10, 8, 4, 50, 80),       # the last size of the logits on this kernel
    (1, 8, 260, 65, 63),      # the first size past the aggregation's
])
def test_small_separate_operators(dtype, B, d, C, H, W):
    """qk and av around the sizes where they change kernels: fp32 bit for bit the reference order's
    sums (the C oracle); 16-bit results within one rounding of the fp32 call on the same values."""
    import sapa_amd
    from oracle import c_oracle
    g = torch.Generator().manual_seed(W)
    q, k, v = (torch.randn(s, generator=g).to(dtype) for s in ((B, d, 2 * H, 2 * W), (B, d, H, W), (B, C, H, W)))
    a = torch.softmax(torch.randn(B, 25, 2 * H, 2 * W, generator=g), dim=1).to(dtype)
    got = sapa_amd.qk(q.cuda(), k.cuda(), 5, 2).cpu(), sapa_amd.av(a.cuda(), v.cuda(), 5, 2).cpu()
    want = c_oracle.qk(q.float(), k.float(), 5, 2, 'f32'), c_oracle.av(a.float(), v.float(), 5, 2, 'f32')
    for x, y in zip(got, want):
        assert torch.equal(x, y) if dtype == torch.float32 else _rel(x, y.double()) <= torch.finfo(dtype).eps / 2 / 3 ** 0.5 * 1.2


@pytest.mark.parametrize('dtype', [torch.float32, torch.bfloat16])
@pytest.mark.parametrize('channels_last', [False, True])
@pytest.mark.parametrize('B,C,O,h,w', [
    (1, 64, 32, 2, 4),         # one chunk per feature
    (2, 256, 64, 100, 168),    # chunks shared by several threads in one feature, a thread per channel in the other
    (3, 512, 32, 24, 20),      # more channels than the threads of a block of few chunks
    # both projections in one launch, a last tile of few pixels each; 2041 tiles, the most for it in fp32; 2198
    (8, 256, 64, 25, 40), (13, 256, 64, 25, 40), (14, 256, 64, 25, 40),
])
def test_norm_project_of_two_features(dtype, channels_last, B, C, O, h, w):
    """sapa_norm_project_pair gives what sapa_norm_project gives for each feature.  (Where one feature
    has many chunks the other's few are added by the same thread either way: bit for bit.)"""
    from sapa_amd import _lib
    g = torch.Generator(device='cuda').manual_seed(C)
    fmt = torch.channels_last if channels_last else torch.contiguous_format
    y, x = (torch.randn(B, C, a, b, generator=g, device='cuda').add_(0.3).to(dtype).contiguous(memory_format=fmt)
            for a, b in ((2 * h, 2 * w), (h, w)))
    norms = [torch.nn.GroupNorm(32, C).cuda().to(dtype) for _ in 'yx']
    convs = [torch.nn.Conv2d(C, O, 1).cuda().to(dtype) for _ in 'yx']
    with torch.no_grad():
        for m in norms:
            m.weight.add_(torch.randn(C, generator=g, device='cuda').to(dtype) * 0.1)
        for defer in (False, True):
            (q, qb), k = _lib.norm_project_pair(y, norms[0], convs[0], x, norms[1], convs[1], channels_last, defer)
            want_q, want_qb = _lib.norm_project(y, norms[0], convs[0], channels_last, defer)
            want_k, _ = _lib.norm_project(x, norms[1], convs[1], channels_last)
            assert torch.equal(q, want_q) and torch.equal(k, want_k)
            assert qb is None and want_qb is None if not defer else torch.equal(qb, want_qb)


@pytest.mark.parametrize('channels_last', [False, True])
def test_plain_projection_keeps_forward_mode_tangents(channels_last):
    """A plain projection in channels_last order of a dual feature under no_grad: the tangent is the
    projection of the feature's tangent (linear up to the bias), within an error bound of a C-term
    fp32 dot product."""
    from torch.autograd import forward_ad
    from sapa_amd.modules import norm_project
    g = torch.Generator(device='cuda').manual_seed(0)
    fmt = torch.channels_last if channels_last else torch.contiguous_format
    x, t = (torch.randn(2, 64, 8, 12, generator=g, device='cuda').contiguous(memory_format=fmt) for _ in 'xt')
    conv = torch.nn.Conv2d(64, 128, 1).cuda()
    with torch.no_grad(), forward_ad.dual_level():
        (out,) = norm_project(forward_ad.make_dual(x, t), None, conv, channels_last=True)
        got = forward_ad.unpack_dual(out).tangent
    assert got is not None
    w = conv.weight.detach().double().reshape(128, 64)
    want = (t.double().permute(0, 2, 3, 1) @ w.T).permute(0, 3, 1, 2)
    mag = (t.double().abs().permute(0, 2, 3, 1) @ w.abs().T).permute(0, 3, 1, 2)
    assert bool(((got.double() - want).abs() <= (64 + 8) * 2.0 ** -24 * mag).all())
