"""CPU: which sizes the two-kernel backward of 16-bit SAPA-B serves."""
import pytest
import torch

from sapa_amd import _lib


@pytest.mark.parametrize('dtype', [torch.float16, torch.bfloat16])
def test_planes_whose_offsets_would_wrap_are_refused(dtype):
    """The kernels stage 16 channels at a time with 32-bit offsets: with fewer channels than that the
    ones past the tensor's last must not come round to its first."""
    serves = _lib.lib().sapa_fused_backward_direct_serves
    code = _lib.DTYPES[dtype]
    # planes of 256 MiB: 16 of them are 2^32 bytes, 8 of them 2^31
    for channels, H, W, contiguous in ((7, 4096, 8192, True), (8, 4096, 8192, False), (7, 4098, 8192, False),
                                       (1, 4096, 8192, True), (1, 4098, 8192, False), (1, 16384, 16382, False),
                                       (17, 1024, 8192, True), (31, 1024, 8192, True), (32, 1024, 8192, False)):
        assert serves(channels, 1, H, W, 5, 2, 0, code) == contiguous, (channels, H, W)
        assert serves(1, channels, H, W, 5, 2, 0, code) == contiguous, (channels, H, W)


def test_norm_project_says_what_it_serves():
    """Asked before anything is allocated: the configurations for which sapa_norm_project has every
    step, by sizes, types and memory orders alone."""
    serves = _lib.lib().sapa_norm_project_serves
    f32, f16, f64 = (_lib.DTYPES[t] for t in (torch.float32, torch.float16, torch.float64))
    for args, expected in (((16, 256, 64, 4200, 32, 0, 0, f32), 1), ((16, 256, 64, 4200, 32, 0, 0, f64), 0),
                           ((1, 512, 64, 1680, 32, 0, 0, f16), 0), ((1, 512, 64, 1680, 32, 1, 1, f16), 1),
                           ((8, 64, 32, 169, 32, 0, 0, f32), 0), ((8, 64, 32, 169, 32, 0, 1, f32), 1),
                           ((8, 64, 32, 172, 32, 0, 1, f16), 0), ((8, 64, 32, 176, 32, 0, 1, f16), 1),
                           ((8, 64, 32, 176, 24, 0, 1, f16), 0), ((1024, 64, 32, 176, 32, 0, 1, f16), 0),
                           ((1024, 64, 32, 176, 32, 1, 1, f16), 1), ((0, 64, 32, 176, 32, 1, 1, f16), 0)):
        assert serves(*args) == expected, args


def test_plain_projections_say_what_extents_they_take():
    """Asked before anything else of a call that the projection kernels would refuse."""
    for dtype, H, W, O, expected in ((torch.bfloat16, 21, 13, 128, False), (torch.bfloat16, 42, 26, 128, False),
                                     (torch.float16, 42, 28, 128, True), (torch.float16, 42, 28, 100, False),
                                     (torch.float32, 42, 26, 128, True), (torch.float32, 21, 13, 128, False)):
        assert _lib.projects_planes(torch.empty(2, 16, H, W, dtype=dtype), O) == expected, (dtype, H, W, O)
