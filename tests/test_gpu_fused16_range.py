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


@pytest.mark.parametrize('channels_last', [False, True])
@pytest.mark.parametrize('scale_q,scale_k,scale_v,scale_go', [
    (0.05, 0.05, 10.0, 3000.0),     # loss-scaled gradients of features that are not normalised: |E| beyond 65504
    (0.0005, 100.0, 10.0, 0.2),     # large keys
    (0.05, 8.0, 1.0, 2.0 ** -13),   # gradients of E below the smallest normal number, lifted by the keys
    (4.0, 1e-2, 1.0, 2.0 ** -15),   # ... by the queries
])
def test_fp16_backward_at_the_ends_of_the_range(channels_last, scale_q, scale_k, scale_v, scale_go):
    """The gradient of the logits leaves fp16's range in both directions while the gradients themselves
    are within it.  Every gradient within one rounding of its own value (2^-11, and half the spacing of
    the subnormals) and an fp32 error (2e-5) of the sum of the magnitudes that it adds up."""
    import sapa_amd
    g = torch.Generator(device='cuda').manual_seed(7)
    B, d, C, H, W = 2, 32, 256, 14, 22
    shapes = ((B, d, 2 * H, 2 * W), (B, d, H, W), (B, C, H, W), (B, C, 2 * H, 2 * W))
    *ops, go = (draw(g, s, torch.float16, f, channels_last) for s, f in zip(shapes, (scale_q, scale_k, scale_v, scale_go)))
    assert go.abs().max() < 20000
    want = exact_gradients(ops, go)[1:]
    # magnitudes: A, |E| and their products with |key|, |query|, |grad_out|
    q, k, v, o = (t.double().contiguous() for t in (*ops, go))
    a = torch.softmax(sapa_amd.qk(q, k, 5, 2), dim=1)
    ga = sapa_amd.qk(o, v, 5, 2)
    scale_e = a * (sapa_amd.qk(o.abs(), v.abs(), 5, 2) + (a * ga.abs()).sum(dim=1, keepdim=True))
    leaves = [t.detach().clone().requires_grad_() for t in (q.abs(), k.abs())]
    mags = list(torch.autograd.grad(sapa_amd.qk(*leaves, 5, 2), leaves, scale_e))
    leaf = v.clone().requires_grad_()
    mags += torch.autograd.grad(sapa_amd.av(a, leaf, 5, 2), leaf, o.abs())
    for got, w, m in zip(gradients(ops, go), want, mags):
        assert w.abs().max() < 65504 and bool(torch.isfinite(got).all())
        bad = (got.double() - w).abs() > 2.0 ** -11 * w.abs() + 2.0 ** -25 + 2e-6 * m
        assert int(bad.sum()) == 0, (int(bad.sum()), bad.numel())


@pytest.mark.parametrize('K,s,W', [(5, 2, 24), (5, 2, 23), (5, 2, 6), (7, 4, 13), (5, 4, 12), (3, 2, 21)])
def test_fp16_forward_of_small_weights(K, s, W):
    """Weights below fp16's smallest normal number on values in the thousands, next to large weights on
    small values: every result within one rounding and an fp32 error of the sum of its terms'
    magnitudes."""
    import sapa_amd
    g = torch.Generator(device='cuda').manual_seed(W)
    B, d, C, H = 2, 32, 16, 9
    q, k = draw(g, (B, d, s * H, s * W), torch.float16, 1.5), draw(g, (B, d, H, W), torch.float16, 1.5)
    v = draw(g, (B, C, H, W), torch.float16, 1.0)
    v = v * torch.where(torch.rand(v.shape, generator=g, device='cuda') < 0.2, 8192.0, 2.0 ** -4).half()
    with torch.no_grad():
        got = sapa_amd.sapa_fused(q, k, v, K, s)
        want = sapa_amd.sapa_fused(q.double(), k.double(), v.double(), K, s)
        mag = sapa_amd.sapa_fused(q.double(), k.double(), v.double().abs(), K, s)
    # (fp32 logits of magnitude 100 are off by 1e-5: so are the weights, relative to themselves)
    bad = (got.double() - want).abs() > 2.0 ** -11 * want.abs() + 2.0 ** -25 + 1e-5 * mag
    assert int(bad.sum()) == 0, (int(bad.sum()), bad.numel())


@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16])
@pytest.mark.parametrize('K,s,H,W', [(5, 2, 3, 33), (5, 2, 5, 7), (7, 4, 3, 21), (5, 4, 5, 9), (3, 2, 3, 33)])
@pytest.mark.parametrize('B', [1, 2, 3])
def test_forward_reads_nothing_behind_a_tensor(K, s, H, W, B, dtype):
    """Tensors of an odd number of elements that end in the middle of a dword, NaN behind them."""
    import sapa_amd
    g = torch.Generator(device='cuda').manual_seed(W)
    d, C = 17, 33

    def tail_nan(shape):
        n = torch.Size(shape).numel()
        buf = torch.full((n + 64,), float('nan'), dtype=dtype, device='cuda')
        buf[:n] = (torch.randn(n, generator=g, device='cuda') * 0.5).to(dtype)
        return buf[:n].view(shape)
    ops = [tail_nan(sh) for sh in ((B, d, s * H, s * W), (B, d, H, W), (B, C, H, W))]
    with torch.no_grad():
        got = sapa_amd.sapa_fused(*ops, K, s)
        again = sapa_amd.sapa_fused(*[t.clone() for t in ops], K, s)
        want = sapa_amd.sapa_fused(*[t.double() for t in ops], K, s)
    assert torch.equal(got, again) and rel(got, want) <= one_rounding(dtype)


def same_non_finite(got, want):
    return (torch.equal(got.isnan(), want.isnan())
            and torch.equal(got == float('inf'), want == float('inf')) and torch.equal(got == -float('inf'), want == -float('inf')))


@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16])
@pytest.mark.parametrize('value', [float('nan'), float('inf')])
@pytest.mark.parametrize('which', [0, 1, 2])
@pytest.mark.parametrize('K,s,W', [(5, 2, 24), (5, 2, 39), (5, 2, 9), (7, 4, 13), (5, 4, 22), (3, 2, 21)])
def test_forward_keeps_non_finite_values_where_they_belong(K, s, W, which, value, dtype):
    """One non-finite element of the query, the key or the value (inside the image and at both ends of a
    row) reaches the results of the windows that hold it and no others."""
    import sapa_amd
    g = torch.Generator(device='cuda').manual_seed(W)
    B, d, C, H = 2, 24, 40, 11
    ops = [draw(g, sh, dtype, 0.5) for sh in ((B, d, s * H, s * W), (B, d, H, W), (B, C, H, W))]
    ops[which][0, 3, 5, 0] = value
    ops[which][1, 7, ops[which].shape[2] - 1, ops[which].shape[3] - 1] = value
    ops[which][1, 2, 4, 7] = -value
    with torch.no_grad():
        got = sapa_amd.sapa_fused(*ops, K, s)
        want = sapa_amd.sapa_fused(*[t.double() for t in ops], K, s)
    assert same_non_finite(got, want)
    ok = torch.isfinite(want)
    assert rel(got[ok], want[ok]) <= one_rounding(dtype)


@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16])
@pytest.mark.parametrize('value', [float('nan'), float('inf')])
@pytest.mark.parametrize('which', [0, 1, 2, 3])
@pytest.mark.parametrize('channels_last,W', [(False, 24), (False, 38), (True, 23)])
def test_backward_keeps_non_finite_values_where_they_belong(channels_last, W, which, value, dtype):
    g = torch.Generator(device='cuda').manual_seed(W)
    B, d, C, H = 2, 24, 40, 11
    shapes = ((B, d, 2 * H, 2 * W), (B, d, H, W), (B, C, H, W), (B, C, 2 * H, 2 * W))
    ops = [draw(g, sh, dtype, 0.5, channels_last) for sh in shapes]
    ops[which][0, 3, 5, 0] = value
    ops[which][1, 7, ops[which].shape[2] - 1, ops[which].shape[3] - 1] = value
    ops[which][1, 2, 4, 7] = -value
    for got, want in zip(gradients(ops[:3], ops[3]), exact_gradients(ops[:3], ops[3])[1:]):
        assert same_non_finite(got, want)
        ok = torch.isfinite(want)
        assert rel(got[ok], want[ok]) <= one_rounding(dtype)


@pytest.mark.parametrize('dtype', [torch.float32, torch.bfloat16, torch.float16])
def test_kept_weights_are_the_ones_the_gradients_come_from(dtype):
    """save_attention=True: the backward pass reads the weights that the forward pass kept (handed back
    as zeros they leave no gradient), and without the option 16-bit tensors keep none."""
    import sapa_amd
    g = torch.Generator(device='cuda').manual_seed(0)
    B, d, C, H, W = 2, 16, 24, 13, 22
    shapes = ((B, d, 2 * H, 2 * W), (B, d, H, W), (B, C, H, W), (B, C, 2 * H, 2 * W))
    *ops, go = (draw(g, sh, dtype, 0.5) for sh in shapes)
    kept = (B, 25, 2 * H, 2 * W)
    for save, expected in ((True, True), (False, False), (None, dtype == torch.float32)):
        leaves, seen = [t.clone().requires_grad_() for t in ops], []
        with torch.autograd.graph.saved_tensors_hooks(lambda t: t, lambda t: seen.append(tuple(t.shape)) or (t * 0 if tuple(t.shape) == kept else t)):
            out = sapa_amd.sapa_fused(*leaves, 5, 2, save_attention=save)
            grads = torch.autograd.grad(out, leaves, go)
        assert (kept in seen) == expected
        assert all(bool((t == 0).all()) for t in grads) == expected


@pytest.mark.parametrize('channels_last', [False, True])
def test_moments_of_two_features_with_an_odd_low_res_plane(channels_last):
    """fp32 features whose low-res planes are no multiple of a vector, into a channels-last module: the
    high-res feature's moments are what they are by themselves, bit for bit."""
    from sapa_amd import _lib
    g = torch.Generator(device='cuda').manual_seed(0)
    C = 64
    y, x = (torch.randn(3, C, a, a, generator=g, device='cuda').contiguous(memory_format=ORDERS[channels_last]) for a in (26, 13))
    norms = [torch.nn.GroupNorm(32, C).cuda() for _ in 'yx']
    convs = [torch.nn.Conv2d(C, 32, 1).cuda() for _ in 'yx']
    with torch.no_grad():
        (q, _), k = _lib.norm_project_pair(y, norms[0], convs[0], x, norms[1], convs[1], True, False)
        assert torch.equal(q, _lib.norm_project(y, norms[0], convs[0], True)[0])
        assert torch.equal(k, _lib.norm_project(x, norms[1], convs[1], True)[0])


def test_an_infinite_feature_in_the_plain_projections():
    """sapa_project_shared in fp32 with infinite and NaN features: infinite and NaN where a 1x1
    convolution is, finite everywhere else."""
    import torch.nn.functional as F
    from sapa_amd import _lib
    g = torch.Generator(device='cuda').manual_seed(0)
    for C, O, H, W in ((64, 40, 9, 12), (256, 128, 16, 20)):
        x = torch.randn(2, C, H, W, generator=g, device='cuda')
        w = torch.randn(O, C, 1, 1, generator=g, device='cuda').mul(0.25)
        w[::2] = w[::2].bfloat16().float()      # weights whose lower pieces are zeros
        x[0, 3, 2, 5], x[0, 5, 8, 11], x[1, 7, 0, 0], x[1, 9, 4, 4], x[1, 10, 4, 4] = (float(t) for t in ('inf', '-inf', 'nan', 'inf', '-inf'))
        x[1, 11, 6, 6] = 3.4e38
        b = torch.randn(O, generator=g, device='cuda')
        want = F.conv2d(x.double(), w.double(), b.double())
        for fmt in ORDERS.values():
            got = _lib.project_shared(x.contiguous(memory_format=fmt), w, b, channels_last_out=fmt == torch.channels_last)
            assert same_non_finite(got, want)
            ok = want.isfinite()
            assert bool(((got[ok].double() - want[ok]).abs() <= 1e-5 + 1e-5 * want[ok].abs()).all())


@pytest.mark.parametrize('channels_last', [False, True])
@pytest.mark.parametrize('C,O', [(64, 128), (128, 72), (256, 288), (512, 128)])
@pytest.mark.parametrize('mean', [0.0, 1.0])
def test_precision_of_the_plain_fp32_projections(C, O, mean, channels_last):
    """sapa_project_shared in fp32: an error like that of one fp32 sum per 32 channels, C / 32 + 2
    roundings that do not know of each other (a library's convolution is off by 0.9 to 2.8e-7 at these
    sizes)."""
    from sapa_amd import _lib
    g = torch.Generator(device='cuda').manual_seed(C)
    B, H, W = 2, 64, 64
    x = (torch.randn(B, C, H, W, generator=g, device='cuda') + mean).contiguous(memory_format=ORDERS[channels_last])
    w = torch.randn(O, C, 1, 1, generator=g, device='cuda').mul(0.02)
    b = torch.randn(O, generator=g, device='cuda').mul(0.1)
    want = torch.matmul(w.double().reshape(O, C), x.double().contiguous().reshape(B, C, H * W)).view(B, O, H, W) + b.double().view(1, O, 1, 1)
    assert rel(_lib.project_shared(x, w, b, channels_last_out=channels_last), want) <= 2.0 ** -24 * (C / 32 + 2) ** 0.5


@pytest.mark.parametrize('C,H,W,aggregated', [(512, 83, 85, False), (512, 85, 85, True), (512, 129, 133, True),
                                              (512, 131, 133, False), (512, 85, 86, False), (128, 190, 197, False)])
def test_training_output_of_odd_rows_on_both_sides_of_the_rule(C, H, W, aggregated):
    """The output of a training step that keeps its weights: with odd rows and a mid-sized value by the
    aggregation with those weights, else by the one-launch forward, the same bits as without gradients."""
    import sapa_amd
    g = torch.Generator(device='cuda').manual_seed(W)
    d = 16
    ops = [draw(g, sh, torch.bfloat16, 0.5) for sh in ((1, d, 2 * H, 2 * W), (1, d, H, W), (1, C, H, W))]
    got = sapa_amd.sapa_fused(*[t.clone().requires_grad_() for t in ops], 5, 2, save_attention=True).detach()
    with torch.no_grad():
        one_launch = sapa_amd.sapa_fused(*ops, 5, 2)
        want = sapa_amd.sapa_fused(*[t.double() for t in ops], 5, 2)
    assert torch.equal(got, one_launch) != aggregated
    assert rel(got, want) <= one_rounding(torch.bfloat16)


@pytest.mark.parametrize('dtype,B,H,W,kernel', [
    (torch.bfloat16, 1, 8, 32, 'sapa_b_dot2_kernel'), (torch.float16, 4, 85, 104, 'sapa_b_dot2_kernel'),
    (torch.bfloat16, 1, 8, 28, 'sapa_b_mfma_kernel'), (torch.float16, 4, 85, 102, 'sapa_b_mfma_kernel'),
    (torch.float32, 8, 64, 64, 'sapa_b_mfma_kernel'), (torch.float32, 3, 110, 100, 'sapa_b_tiled_kernel'),
    (torch.float32, 3, 110, 101, 'sapa_b_mfma_kernel')])
def test_logits_on_both_sides_of_the_rule(dtype, B, H, W, kernel):
    """qk by the matrix-pipe kernel where the thread-per-parent kernels do not read rows in vectors, and in
    fp32 up to 32768 cells; by the dot-product kernel for 16-bit rows of whole vectors."""
    import sapa_amd
    from sapa_amd import _lib
    g = torch.Generator(device='cuda').manual_seed(W)
    d = 32
    q, k = draw(g, (B, d, 2 * H, 2 * W), dtype, 0.5), draw(g, (B, d, H, W), dtype, 0.5)
    with torch.no_grad():
        got = sapa_amd.qk(q, k, 5, 2)
        assert _lib.last_kernel().startswith(kernel)
        want = sapa_amd.qk(q.double(), k.double(), 5, 2)
    # (32 fp32 roundings that do not know of each other, or one to the result's type)
    assert rel(got, want) <= (one_rounding(dtype) if dtype != torch.float32 else 32 ** 0.5 * 2.0 ** -24)
