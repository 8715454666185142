"""Bias gradient of small planes in one launch (csrc/crb_conv.hip, bias_grad_one_kernel) where its blocks end: planes of every
size it takes, channels that fill no block of 64 columns, row slices of every count; beside it planes that keep two launches."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(1, 2, 2), (7, 33, 4), (128, 512, 4), (16, 5, 16), (130, 512, 16), (33, 6, 64), (512, 64, 64), (127, 3, 128), (128, 128, 256),
                                   (129, 2, 256), (8, 3, 1024), (6, 5, 36)], ids=lambda s: "x".join(map(str, s)))
def test_bias_gradient_of_small_planes(dev, shape):
    import torch
    from crusaderbackend_amd import capi

    N, C, HW = shape
    dY, dB0 = torch.randn(N, C, HW, device=dev), torch.randn(C, device=dev)
    got = [dB0.clone() for _ in range(2)]
    for dB in got:
        capi.conv_bias_grad(dY, dB, N, C, HW)
    # the same rows one float off the 16-byte grid run in two launches
    off = torch.empty(dY.numel() + 1, device=dev)
    off[1:].copy_(dY.view(-1))
    two = dB0.clone()
    capi.conv_bias_grad(off[1:], two, N, C, HW)
    torch.cuda.synchronize()
    ref, size = dB0.cpu().double() + dY.cpu().double().sum((0, 2)), dB0.cpu().double().abs() + dY.cpu().double().abs().sum((0, 2))
    assert torch.equal(*got)
    # rows, 16 row lanes, slices and the plane's tree: at most N / 16 + 32 additions in a row, each off by 2^-24 of the sum so far
    for dB in (got[0], two):
        assert ((dB.cpu().double() - ref).abs() <= (N / 16 + 32) * 2.0**-24 * size).all()
