"""1x1 layers on few images run on small tiles (csrc/crb_conv.hip, try_pointwise): extents, channel counts and batches on either
side of where the configurations change, against float64."""
import pytest

pytestmark = pytest.mark.gpu

# (N, IC, OC, H, W)
LAYERS = [(2, 17, 33, 32, 32), (16, 204, 48, 32, 32), (42, 30, 48, 32, 32), (43, 30, 48, 32, 32), (48, 100, 13, 24, 32), (5, 385, 20, 16, 32), (3, 384, 20, 4, 32),
          (3, 191, 47, 16, 16), (3, 192, 47, 16, 16), (42, 33, 48, 16, 16), (43, 33, 48, 16, 16), (8, 330, 48, 8, 8), (7, 20, 150, 24, 8), (86, 40, 40, 8, 8),
          (1, 249, 60, 24, 16), (2, 9, 12, 20, 16)]


@pytest.mark.parametrize("layer", LAYERS, ids=lambda l: "x".join(map(str, l)))
def test_small_batches_of_pointwise_layers(dev, layer):
    import torch
    from crusaderbackend_amd import capi

    N, IC, OC, H, W = layer
    g = capi.ConvGeom.make(N, IC, H, W, OC, 1, 1)
    X, dY, Wt, b = (torch.randn(*s, device=dev) for s in ((N, IC, H, W), (N, OC, H, W), (OC, IC), (OC,)))
    Y, dX = torch.empty_like(dY), torch.empty_like(X)
    capi.conv_fwd(Wt, X, Y, b, g, capi.CRB_FLAG_RELU)
    capi.conv_dgrad(Wt, dY, dX, g)
    torch.cuda.synchronize()
    w = Wt.cpu().double()
    y = (w @ X.cpu().double().view(N, IC, -1) + b.cpu().double()[:, None]).relu().view(N, OC, H, W)
    dx = (w.t().contiguous() @ dY.cpu().double().view(N, OC, -1)).view(N, IC, H, W)
    # every product and sum rounds once: 0.29 * 2^-23 of a partial sum, 0.71 of the last one in the mean, and the bias
    assert (Y.cpu().double() - y).norm() <= (IC + 2) ** 0.5 * 2.0**-25 * y.norm() * 2
    assert (dX.cpu().double() - dx).norm() <= OC**0.5 * 2.0**-25 * dx.norm() * 2
