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
