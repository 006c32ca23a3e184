"""The work that a user of these operators has them do, as cases that can be timed.

A case is one call of the public API at one size: `kind` says which call, the other entries its
extents, element type and memory order.

  ops            attn = softmax(qk(q, k)); out = av(attn, v): the separate operators
  fused          sapa_fused(q, k, v) without gradients
  module         SAPA(...)(y, x) without gradients, the norms folded into the projections
  train          sapa_fused forward and backward: the output and the gradients of q, k and v
  deform_fused   deform_sapa_fused(q, k, v, offset) without gradients
  deform_module  SAPADeform(...)(y, x) without gradients
  deform_train   deform_sapa_fused forward and backward: the output and all four gradients

H, W are the low-res extents; the output has s*H x s*W pixels.
"""
import math

import torch
import torch.nn.functional as F

import sapa_amd

DTYPES = {'fp32': torch.float32, 'fp16': torch.float16, 'bf16': torch.bfloat16}


def _case(name, kind, dtype, layout, B, C, d, H, W, K=5, s=2, P=0, G=0):
    case = dict(kind=kind, dtype=dtype, layout=layout, B=B, C=C, d=d, H=H, W=W, s=s)
    case.update(dict(P=P, G=G) if P else dict(K=K))
    return dict(case, name=name) if name else case


def listed():
    return [
        # one image through the separate operators, the reference's own composition: the smallest
        # call there is, launches and host time
        _case('ops_single_fp32', 'ops', 'fp32', 'nchw', 1, 64, 32, 32, 32),
        # the first decoder stage of a SegFormer segmentation head at inference (stride 32 -> 16)
        _case('module_segformer_16_bf16', 'module', 'bf16', 'nchw', 8, 256, 32, 16, 16),
        # the coarsest FPN level of a batch of portrait 1333 x 800 images: an odd width
        _case('fused_fpn_small_portrait_bf16', 'fused', 'bf16', 'nchw', 16, 256, 64, 42, 25),
        # the largest FPN level of a batch of 800 x 1333 images in fp32, contiguous tensors: what
        # the reference's own detection models run at inference
        _case('fused_fpn_large_fp32', 'fused', 'fp32', 'nchw', 16, 256, 64, 100, 168),
        # the middle FPN level as a module in fp32, features as a reference model holds them
        _case('module_fpn_mid_fp32', 'module', 'fp32', 'nchw', 16, 256, 64, 50, 84),
        # the largest FPN level as a module in a channels-last bf16 model (served inference)
        _case('module_fpn_large_bf16_cl', 'module', 'bf16', 'channels_last', 16, 256, 64, 100, 168),
        # one step x4 up with a 7 x 7 window on 512 channels: the heaviest window in use
        _case('fused_k7_s4_bf16', 'fused', 'bf16', 'nchw', 4, 512, 64, 64, 64, K=7, s=4),
        # training of the largest FPN level under bf16 autocast, contiguous tensors
        _case('train_fpn_large_bf16', 'train', 'bf16', 'nchw', 16, 256, 64, 100, 168),
        # training of the middle FPN level in fp32, the reference's training precision
        _case('train_fpn_mid_fp32', 'train', 'fp32', 'nchw', 16, 256, 64, 50, 84),
        # training of the last SegFormer stage in a channels-last fp16 model (mixed precision)
        _case('train_segformer_64_fp16_cl', 'train', 'fp16', 'channels_last', 8, 256, 32, 64, 64),
        # SAPA-D with the reference's default 9 points as a module in fp32
        _case('deform_module_p9_fp32', 'deform_module', 'fp32', 'nchw', 8, 256, 32, 64, 64, P=9, G=4),
        # SAPA-D training with 25 points in bf16
        _case('deform_train_p25_bf16', 'deform_train', 'bf16', 'nchw', 8, 256, 32, 64, 64, P=25, G=4),
    ]


def draw(rng):
    """One more case of the same ranges: any call, type and memory order in use, extents from one
    16 x 16 image to the largest FPN level of 16, odd widths and heights among them."""
    kind = rng.choice(['ops', 'fused', 'fused', 'module', 'module', 'train', 'train', 'train',
                       'deform_fused', 'deform_module', 'deform_train'])
    dtype = rng.choice(['fp32', 'bf16', 'bf16', 'fp16'])
    layout = 'nchw' if kind == 'ops' else rng.choice(['nchw', 'nchw', 'channels_last'])
    deform = kind.startswith('deform')
    C = rng.choice([64, 128, 256, 256, 512])
    d = 32 if deform else rng.choice([32, 64])
    B = round(math.exp(rng.uniform(0, math.log(16))))
    # low-res cells of the whole batch; SAPA-D is used at the smaller levels
    cells = math.exp(rng.uniform(math.log(1024), math.log(65536 if deform else 262144))) / (C / 256)
    aspect = math.exp(rng.uniform(math.log(0.55), math.log(1.8)))
    area = max(256.0, cells / B)
    H = min(192, max(13, round(math.sqrt(area / aspect))))
    W = min(192, max(13, round(math.sqrt(area * aspect))))
    B = max(1, min(B, int(262144 * 256 / (C * H * W))))
    if deform:
        return _case(None, kind, dtype, layout, B, C, d, H, W, P=rng.choice([5, 9, 9, 25]), G=4)
    K, s = 5, 2
    if kind == 'fused' and rng.random() < 0.25:
        K, s = rng.choice([(3, 2), (7, 2), (5, 4), (7, 4)])
        if s == 4:
            H, W = max(8, H // 2), max(8, W // 2)
    return _case(None, kind, dtype, layout, B, C, d, H, W, K=K, s=s)


def prepare(case, seed):
    dev, dtype = torch.device('cuda'), DTYPES[case['dtype']]
    fmt = torch.channels_last if case['layout'] == 'channels_last' else torch.contiguous_format
    g = torch.Generator(device=dev).manual_seed(seed)
    B, C, d, H, W, s = (case[k] for k in ('B', 'C', 'd', 'H', 'W', 's'))
    kind = case['kind']
    deform = kind.startswith('deform')

    def feature(channels, h, w):
        return torch.randn(B, channels, h, w, generator=g, device=dev)

    def as_used(t):
        return t.to(dtype).contiguous(memory_format=fmt)
    state = dict(case)
    if kind in ('module', 'deform_module'):
        # features behind a ReLU backbone's lateral convolutions: zero mean, channels of unequal size
        y = feature(C, s * H, s * W) * (0.5 + torch.rand(1, C, 1, 1, generator=g, device=dev))
        x = feature(C, H, W) * (0.5 + torch.rand(1, C, 1, 1, generator=g, device=dev))
        state['y'], state['x'] = as_used(y), as_used(x)
        options = dict(up_factor=s, embedding_dim=d, channels_last=case['layout'] == 'channels_last')
        if deform:
            m = sapa_amd.SAPADeform(C, num_point=case['P'], groups=case['G'], **options)
        else:
            m = sapa_amd.SAPA(C, up_kernel_size=case['K'], fold_norm=True, **options)
        m = m.to(dev)
        with torch.no_grad():
            for name, p in m.named_parameters():
                draws = torch.randn(p.shape, generator=g, device=dev)
                if p.dim() == 4:
                    p.copy_(draws * 0.02)
                else:
                    p.copy_(draws * 0.1 + (1.0 if name.startswith('norm') and name.endswith('weight') else 0.0))
        state['module'] = m.to(dtype).eval().requires_grad_(False)
        return state
    groups = case['G'] if deform else 1
    # queries and keys as 1x1 projections give them: zero mean, key channels of unequal size
    q = feature(groups * d, s * H, s * W) * 0.5
    k = feature(groups * d, H, W) * (0.25 + 0.5 * torch.rand(1, groups * d, 1, 1, generator=g, device=dev))
    v = feature(C, H, W)
    tensors = [q, k, v]
    if deform:
        tensors.append((0.75 * feature(2 * groups * case['P'], s * H, s * W)).clamp(-4, 4))
    tensors = [as_used(t) for t in tensors]
    if kind.endswith('train'):
        state['grad'] = as_used(feature(C, s * H, s * W))
        tensors = [t.requires_grad_() for t in tensors]
    state['tensors'] = tensors
    return state


def run(state):
    kind, s = state['kind'], state['s']
    if kind in ('module', 'deform_module'):
        with torch.no_grad():
            return state['module'](state['y'], state['x'])
    if kind == 'ops':
        q, k, v = state['tensors']
        attn = F.softmax(sapa_amd.qk(q, k, state['K'], s), dim=1)
        return sapa_amd.av(attn, v, state['K'], s)
    if kind.startswith('deform'):
        out = sapa_amd.deform_sapa_fused(*state['tensors'], state['P'], s, state['G'])
    else:
        out = sapa_amd.sapa_fused(*state['tensors'], state['K'], s)
    if not kind.endswith('train'):
        return out
    return (out.detach(),) + torch.autograd.grad(out, state['tensors'], state['grad'])


def work(case):
    """Every input read once, every output written once; the multiply-adds of the operators (and
    of the projections), and twice as many again for their gradients."""
    kind, esize = case['kind'], 4 if case['dtype'] == 'fp32' else 2
    B, C, d, H, W, s = (case[k] for k in ('B', 'C', 'd', 'H', 'W', 's'))
    lo, hi = B * H * W, B * H * W * s * s
    if kind.startswith('deform'):
        G, P = case['G'], case['P']
        dq, doff = G * d, 2 * G * P
        flops = hi * 2 * 5 * P * (dq + C)
    else:
        dq, doff = d, 0
        flops = hi * 2 * case['K'] ** 2 * (d + C)
    if kind in ('module', 'deform_module'):
        elements = (hi + lo) * C + hi * C
        flops += 2 * C * ((hi + lo) * dq + lo * doff * s * s)
    elif kind.endswith('train'):
        # read: the operands and the gradient of the output; written: the output and the gradients
        elements = 2 * (hi * (dq + doff + C) + lo * (dq + C))
        flops *= 3
    else:
        elements = hi * (dq + doff + C) + lo * (dq + C)
    return {'bytes': elements * esize, 'flops': flops}


# Largest relative error (2-norm) of an output against the same call in float64 on the same
# inputs, about four times the largest measured over the listed sizes and a dozen drawn ones
# (fp32 3e-7 to 5e-7, SAPA-D 9e-7 forward and 4e-6 for gradients; fp16 2.1e-4, bf16 1.7e-3, one
# rounding of the result; where a 16-bit tensor stands between two calls -- the weights between
# qk and av, the projected queries and keys -- twice to three times that).  The gradient of the
# offsets jumps where a sampling position crosses a cell: the operators pin that index exactly.
TOLERANCES = {
    'fp32': {'deform_fused': 5e-6, 'deform_module': 5e-6, 'deform_train': 2e-5, 'other': 3e-6},
    'fp16': {'ops': 2e-3, 'module': 1.6e-3, 'deform_module': 1.6e-3, 'other': 8.5e-4},
    'bf16': {'ops': 1e-2, 'module': 1e-2, 'deform_module': 1e-2, 'other': 7e-3},
}


def tolerance(case):
    table = TOLERANCES[case['dtype']]
    return {'rel': table.get(case['kind'], table['other'])}
