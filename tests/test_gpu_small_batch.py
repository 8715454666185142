"""Width-specialised 3x3 layers on few images run on smaller tiles (csrc/crb_conv.hip, try_direct): per image the results have the
bits of a large batch, whose tiles and chunks are others."""
import pytest

pytestmark = pytest.mark.gpu

# (IC, H, W, OC), small batches on either side of where the tiles change, a batch on the large tiles
LAYERS = [(64, 32, 32, 64, (1, 2, 4, 5, 16, 17), 130), (72, 32, 32, 40, (8, 20), 140), (128, 16, 16, 128, (3, 8, 39, 40), 66),
          (40, 16, 16, 104, (9, 45), 100), (24, 16, 16, 64, (1, 32), 44), (256, 8, 8, 256, (8, 32, 33, 64), 70), (20, 16, 8, 136, (5, 28), 66),
          (136, 8, 8, 128, (8, 32), 34), (512, 4, 4, 512, (8, 16, 64), 70), (56, 4, 4, 24, (6, 30), 1100)]


@pytest.mark.parametrize("layer", LAYERS, ids=lambda l: "x".join(map(str, l[:4])))
def test_small_batches_have_the_bits_of_large_ones(dev, layer):
    import torch
    from crusaderbackend_amd import capi

    IC, H, W, OC, small, large = layer
    X, dY = torch.randn(large, IC, H, W, device=dev), torch.randn(large, OC, H, W, device=dev)
    Wt, b = torch.randn(OC, IC, 3, 3, device=dev) / (IC * 9) ** 0.5, torch.randn(OC, device=dev)
    # (the data gradient of a layer with the roles of the channels exchanged: the same configurations)
    Wd = torch.randn(IC, OC, 3, 3, device=dev) / (IC * 9) ** 0.5

    def run(n):
        Y, dX = torch.full((n, OC, H, W), float("nan"), device=dev), torch.full((n, OC, H, W), float("nan"), device=dev)
        capi.conv_fwd(Wt, X[:n], Y, b, capi.ConvGeom.make(n, IC, H, W, OC, 3, 3, 1, 1, 1, 1), capi.CRB_FLAG_RELU)
        capi.conv_dgrad(Wd, X[:n], dX, capi.ConvGeom.make(n, OC, H, W, IC, 3, 3, 1, 1, 1, 1))
        torch.cuda.synchronize()
        return Y, dX

    Y, dX = run(large)
    ref = torch.nn.functional.conv2d(X[:2].cpu().double(), Wt.cpu().double(), b.cpu().double(), padding=1).relu()
    assert (Y[:2].cpu().double() - ref).norm() <= 2.0**-24 * (IC * 9) ** 0.5 * ref.norm()
    for n in small:
        y, dx = run(n)
        assert torch.equal(dx, dX[:n]), n
        if n >= 8:  # (fewer: other kernels, conv_few.h and conv_split.h)
            assert torch.equal(y, Y[:n]), n
