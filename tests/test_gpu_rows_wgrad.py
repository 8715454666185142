"""3x3 weight gradients on rows of octets (csrc/conv_split_wgrad_rows.h) where its rows, tiles, slices and channel blocks end."""
import numpy as np
import pytest

from oracle import seblas_oracle as orc
from tests.util import assert_close, launched, normal, to_dev, to_np

pytestmark = pytest.mark.gpu

# (N, IC, H, W, OC, words the operands lie off a 16-byte address): rows of one octet, of 2 pixels, of an octet of which nothing is padding but one, of whole
# octets and of the most there are; loads of four, two and one pixels; the least rows of an image; blocks of channels that end early; one
# slice without a sum behind it and many; a last tile of few octets
SHAPES = [(40, 64, 17, 6, 40, 0), (30, 128, 40, 2, 96, 0), (16, 64, 23, 14, 64, 0), (9, 33, 20, 24, 65, 0), (3, 80, 31, 56, 48, 0), (6, 50, 9, 62, 63, 0),
          (2, 40, 33, 126, 33, 0), (2, 96, 21, 100, 32, 2), (5, 64, 14, 44, 72, 1), (4, 512, 9, 12, 512, 0), (1, 64, 30, 46, 130, 0), (7, 64, 9, 10, 512, 3)]


def arrays(shape, dev):
    N, IC, H, W, OC, off = shape
    X, dY, dW0 = normal(1, N, IC, H, W), normal(2, N, OC, H, W), normal(3, OC, IC, 3, 3)

    def at(a):
        import torch

        t = torch.empty(a.size + off, device=dev)[off:].view(*a.shape)
        return t.copy_(torch.from_numpy(a))

    return X, dY, dW0, at(X), at(dY), to_dev(dW0, dev)


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_rows_weight_gradient_edges(dev, shape):
    import torch
    from crusaderbackend_amd import capi

    N, IC, H, W, OC, off = shape
    g = capi.ConvGeom.make(N, IC, H, W, OC, 3, 3, 1, 1, 1, 1)
    X, dY, dW0, Xd, dYd, dW = arrays(shape, dev)
    capi.conv_wgrad(dYd, Xd, dW, g)
    again = to_dev(dW0, dev)
    capi.conv_wgrad(dYd, Xd, again, g, workspace=torch.empty(capi.conv_wgrad_workspace_bytes(g) // 4 + 1, device=dev))
    torch.cuda.synchronize()
    assert_close(to_np(dW), orc.convError(dY, X, dW0, 1, 1, 1, 1), N * H * W, f"weight gradient {shape}")
    assert torch.equal(dW, again)
    words = 4 if W % 4 == 0 and off % 4 == 0 else 2 if off % 2 == 0 else 1
    kernels = [k for k, _ in launched(dev, lambda stream: capi.conv_wgrad(dYd, Xd, again, g, stream=stream))]
    assert any(f"rows_wgrad_kernelILi{words}E" in k for k in kernels), kernels


@pytest.mark.parametrize("shape", [SHAPES[0], SHAPES[2], SHAPES[3], SHAPES[9]], ids=lambda s: "x".join(map(str, s)))
def test_rows_weight_gradient_of_operands_that_are_not_finite(dev, shape):
    """An infinite pixel at a corner, one inside and a channel of infinities: what float64 gives, the padding between rows and images
    taking no part; elements whose terms are all finite are as close as ever."""
    import torch
    from crusaderbackend_amd import capi

    N, IC, H, W, OC, off = shape
    g = capi.ConvGeom.make(N, IC, H, W, OC, 3, 3, 1, 1, 1, 1)
    X, dY, dW0, Xd, dYd, _ = arrays(shape, dev)
    X, dY = np.abs(X) + 0.25, np.abs(dY) + 0.25  # (no infinity meets one of the other sign, or a zero)
    X[N - 1, IC - 1, H - 1, W - 1] = X[0, 3, 0, 0] = X[0, 7, H // 2, W // 2] = np.inf
    dY[:, OC - 1] = np.inf
    Xd.copy_(torch.from_numpy(X)), dYd.copy_(torch.from_numpy(dY))
    dW = torch.zeros(OC, IC, 3, 3, device=dev)
    capi.conv_wgrad(dYd, Xd, dW, g)
    torch.cuda.synchronize()
    ref = np.zeros((OC, IC, 3, 3))
    with np.errstate(invalid="ignore"):
        for fh in range(3):
            for fw in range(3):
                ys, xs = slice(max(0, 1 - fh), H - max(0, fh - 1)), slice(max(0, 1 - fw), W - max(0, fw - 1))
                yx, xx = slice(max(0, fh - 1), H - max(0, 1 - fh)), slice(max(0, fw - 1), W - max(0, 1 - fw))
                d, x = dY[:, :, ys, xs].astype(np.float64), X[:, :, yx, xx].astype(np.float64)
                finite = np.einsum("noyx,niyx->oi", np.where(np.isinf(d), 0, d), np.where(np.isinf(x), 0, x))
                ref[:, :, fh, fw] = np.where(np.isinf(d).any((0, 2, 3))[:, None] | np.isinf(x).any((0, 2, 3))[None], np.inf, finite)
    got = to_np(dW).astype(np.float64)
    assert np.array_equal(np.isinf(got), np.isinf(ref)) and not np.isnan(got).any()
    ok = np.isfinite(ref)
    assert np.abs(got - ref)[ok].max() <= 1e-5 * np.sqrt(N * H * W) * ref[ok].max()


def test_rows_weight_gradient_is_recorded(dev):
    """In a graph, with a workspace of the queried size, the replays give the eager result."""
    import torch
    from crusaderbackend_amd import capi

    g = capi.ConvGeom.make(9, 64, 20, 24, 65, 3, 3, 1, 1, 1, 1)
    X, dY = torch.randn(9, 64, 20, 24, device=dev), torch.randn(9, 65, 20, 24, device=dev)
    ws = torch.empty(capi.conv_wgrad_workspace_bytes(g) // 4 + 1, device=dev)
    eager, out = (torch.zeros(65, 64, 3, 3, device=dev) for _ in range(2))
    capi.conv_wgrad(dY, X, eager, g, workspace=ws)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=torch.cuda.Stream(device=dev)):
        capi.conv_wgrad(dY, X, out, g, workspace=ws, stream=torch.cuda.current_stream())
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager)
