"""Forward passes of 3x3 layers on a handful of images (csrc/conv_few.h) where its tiles, chunks and slices end: one to seven
images, 2 x 2 images that do not fill a tile of four, channels that fill neither a chunk of 64 nor a block of 16, tiles of
every shape, one slice and several."""
import numpy as np
import pytest

from oracle import seblas_oracle as orc
from tests.util import assert_close, he_normal, normal, to_dev, to_np

pytestmark = pytest.mark.gpu

# (N, IC, H, W, OC)
SHAPES = [(1, 64, 2, 2, 16), (3, 80, 2, 2, 33), (7, 512, 2, 2, 50), (1, 64, 4, 4, 40), (2, 144, 8, 4, 17), (5, 64, 6, 8, 31), (3, 336, 2, 8, 48),
          (1, 96, 3, 16, 64), (2, 128, 7, 32, 24), (1, 512, 4, 4, 512), (1, 64, 5, 48, 130), (7, 1040, 4, 4, 16)]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_few_pixels(dev, shape):
    """Against the oracle and, on random operands, no further from float64 than sums of chains of twelve terms are: a chain's
    roundings are 0.29 * 2^-23 of what is summed so far each, those of K / 12 chains and of the waves and slices the same."""
    import torch
    import torch.nn.functional as F
    from crusaderbackend_amd import capi

    N, IC, H, W, OC = shape
    g = capi.ConvGeom.make(N, IC, H, W, OC, 3, 3, 1, 1, 1, 1)
    X, Wt, b = normal(1, N, IC, H, W), he_normal(2, OC, IC, 3, 3), normal(3, OC)
    Xd, Wd, bd = to_dev(X, dev), to_dev(Wt, dev), to_dev(b, dev)
    Y = torch.empty(N, OC, H, W, device=dev)
    for bias, flags in ((b, capi.CRB_FLAG_RELU), (None, 0)):
        capi.conv_fwd(Wd, Xd, Y, bd if bias is not None else None, g, flags)
        torch.cuda.synchronize()
        ref = orc.conv(Wt, X, bias, 1, 1, 1, 1)
        assert_close(to_np(Y), np.maximum(ref, 0) if flags else ref, IC * 9, f"few pixels {shape}")
    exact = F.conv2d(torch.from_numpy(X).double(), torch.from_numpy(Wt).double(), padding=1)
    assert (Y.cpu().double() - exact).norm() <= np.sqrt(12 + IC * 9 / 12) * 2.0**-25 * exact.norm()

    # less scratch than the slices take: launched one after the other, the same bits
    if need := capi.conv_fwd_workspace_bytes(g):
        again, side, little = torch.empty_like(Y), torch.cuda.Stream(device=dev), torch.empty(need // 4 - 64, device=dev)
        torch.cuda.synchronize()
        try:
            capi.bind_workspace(little, stream=side)
            capi.conv_fwd(Wd, Xd, again, None, g, 0, stream=side)
            side.synchronize()
            assert torch.equal(Y, again)
        except capi.CrbError as e:  # (calls that the fp32 kernel for them would be refused too: not where a width-specialised one stands behind)
            assert e.status == capi.CRB_EWORKSPACE and shape != (1, 512, 4, 4, 512)
        finally:
            capi.bind_workspace(None, stream=side)

    # infinite operands: a filter element outside the image takes no part
    Xi, Wi = Xd.clone(), Wd.clone()
    Xi[0, 1, -1, -1], Xi[N - 1, IC - 1, 0, 0], Wi[OC // 2, 5, 0, 2], Wi[OC - 1, 0, 2, 2] = float("inf"), -3.4e38, float("-inf"), float("inf")
    capi.conv_fwd(Wi, Xi, Y, None, g, 0)
    torch.cuda.synchronize()
    y = _conv64(Xi.cpu().double().numpy(), Wi.cpu().double().numpy())
    np.testing.assert_allclose(to_np(Y), np.where(np.abs(y) > 3.4028235e38, np.copysign(np.inf, y), y), rtol=IC * 9 * 2.0**-23, atol=IC * 9 * 2.0**-20,
                               equal_nan=True)


def _conv64(X, W):
    """Taps outside the image take no part."""
    N, _, H, Wd = X.shape
    y = np.zeros((N, W.shape[0], H, Wd))
    with np.errstate(invalid="ignore"):
        for fh in range(3):
            for fw in range(3):
                ys, xs = slice(max(0, 1 - fh), min(H, H + 1 - fh)), slice(max(0, 1 - fw), min(Wd, Wd + 1 - fw))
                src = X[:, :, ys.start + fh - 1 : ys.stop + fh - 1, xs.start + fw - 1 : xs.stop + fw - 1]
                y[:, :, ys, xs] += sum(W[None, :, c, fh, fw, None, None] * src[:, c][:, None] for c in range(X.shape[1]))
    return y


def test_which_calls_run_on_few_pixels():
    """Seen from the scratch: slices of the result, or none; eight images and more keep what a training step runs."""
    from crusaderbackend_amd import capi

    def need(N, IC, H, OC):
        return capi.conv_fwd_workspace_bytes(capi.ConvGeom.make(N, IC, H, H, OC, 3, 3, 1, 1, 1, 1))

    assert need(1, 512, 4, 512) == 8 * 512 * 16 * 4 and need(8, 512, 4, 512) == 0
    assert need(1, 64, 32, 64) == 0 and need(7, 64, 32, 64) > 6 * 64 * 64 * 9
