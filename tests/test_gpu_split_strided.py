"""Strided layers on split bf16 operands where tiles, strips, chunks and filter rows end: 5x5 stride 2 forward and weight gradient
(csrc/conv_split.h with one place for the run, csrc/conv_split_wgrad.h by filter rows), 3x3 and 5x5 data gradient at stride 2 by residue
classes (csrc/conv_split.h)."""
import numpy as np
import pytest

from oracle import seblas_oracle as orc
from tests.util import assert_close, he_normal, normal, to_dev, to_np

pytestmark = pytest.mark.gpu

# (N, IC, H, W, OC, F, stride, pad): odd and even extents, every padding, channels that fill no chunk or block, one image row, many
# strips, tiles that cross images, a cut contraction
SHAPES = [(24, 30, 61, 47, 75, 5, 2, 2), (3, 31, 41, 39, 133, 5, 2, 1), (40, 50, 13, 12, 70, 5, 2, 4), (2, 90, 5, 151, 97, 5, 2, 0), (9, 233, 11, 13, 150, 5, 2, 2),
          (64, 40, 9, 9, 100, 5, 2, 3), (5, 17, 64, 65, 193, 5, 2, 2), (33, 65, 15, 8, 65, 5, 2, 2),
          (16, 64, 57, 55, 128, 3, 2, 1), (6, 200, 30, 28, 77, 3, 2, 1), (50, 33, 9, 8, 250, 3, 2, 0), (3, 130, 41, 96, 65, 3, 2, 2), (29, 28, 3, 50, 130, 5, 2, 3),
          (90, 300, 7, 7, 90, 3, 2, 1), (200, 24, 2, 31, 120, 3, 2, 1)]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_strided_layers(dev, shape):
    """Against the oracle; the forward pass and both gradients, with less scratch than they take the same bits or a refusal."""
    import torch
    from crusaderbackend_amd import capi

    N, IC, H, W, OC, F, s, p = shape
    g = capi.ConvGeom.make(N, IC, H, W, OC, F, F, s, s, p, p)
    X, Wt, dY, b = normal(1, N, IC, H, W), he_normal(2, OC, IC, F, F), normal(3, N, OC, g.OH, g.OW), normal(4, OC)
    Xd, Wd, dYd, bd = (to_dev(x, dev) for x in (X, Wt, dY, b))
    Y, dX, dW0 = torch.empty(N, OC, g.OH, g.OW, device=dev), torch.empty(N, IC, H, W, device=dev), normal(5, OC, IC, F, F)
    dW = to_dev(dW0, dev)
    capi.conv_fwd(Wd, Xd, Y, bd, g, capi.CRB_FLAG_RELU)
    capi.conv_dgrad(Wd, dYd, dX, g)
    capi.conv_wgrad(dYd, Xd, dW, g)
    torch.cuda.synchronize()
    assert_close(to_np(Y), np.maximum(orc.conv(Wt, X, b, s, s, p, p), 0), IC * F * F, f"fwd {shape}")
    assert_close(to_np(dX), orc.convDerive(Wt, dY, (H, W), s, s, p, p), OC * F * F, f"dgrad {shape}")
    assert_close(to_np(dW), orc.convError(dY, X, dW0, s, s, p, p), N * g.OH * g.OW, f"wgrad {shape}")

    side, again = torch.cuda.Stream(device=dev), (torch.empty_like(Y), torch.empty_like(dX))
    torch.cuda.synchronize()
    for need, call, got, want in ((capi.conv_fwd_workspace_bytes(g), lambda o: capi.conv_fwd(Wd, Xd, o, bd, g, capi.CRB_FLAG_RELU, stream=side), again[0], Y),
                                  (capi.conv_dgrad_workspace_bytes(g), lambda o: capi.conv_dgrad(Wd, dYd, o, g, stream=side), again[1], dX)):
        if need < 1024:
            continue
        little = torch.empty(need // 4 - 128, device=dev)
        torch.cuda.synchronize()
        try:
            capi.bind_workspace(little, stream=side)
            call(got)
            side.synchronize()
            assert torch.equal(got, want)
        except capi.CrbError as e:  # (where the fp32 kernel would be refused too)
            assert e.status == capi.CRB_EWORKSPACE
        finally:
            capi.bind_workspace(None, stream=side)


@pytest.mark.parametrize("shape", [SHAPES[1], SHAPES[4], SHAPES[9], SHAPES[11]], ids=lambda s: "x".join(map(str, s)))
def test_strided_layers_with_infinities(dev, shape):
    """Infinite operands and ones that round to infinity in 16 bits give what sums in fp32 give."""
    import torch
    import torch.nn.functional as F_
    from crusaderbackend_amd import capi

    N, IC, H, W, OC, F, s, p = shape
    g = capi.ConvGeom.make(N, IC, H, W, OC, F, F, s, s, p, p)
    X, Wt, dY = (torch.randn(*d, device=dev) for d in ((N, IC, H, W), (OC, IC, F, F), (N, OC, g.OH, g.OW)))
    Wt /= (IC * F * F) ** 0.5
    X[0, 1, -1, -1], X[N - 1, 3, 0, 0], X[N // 2, IC - 1, H // 2, W // 2] = float("inf"), -3.4e38, float("nan")
    dY[0, 2, 1, 1], dY[N - 1, OC - 1, -1, -1] = float("-inf"), 3.4e38
    Y, dX, dW = torch.empty_like(dY), torch.empty_like(X), torch.zeros_like(Wt)
    capi.conv_fwd(Wt, X, Y, None, g)
    capi.conv_dgrad(Wt, dY, dX, g)
    capi.conv_wgrad(dY, X, dW, g)
    torch.cuda.synchronize()
    x, w, d = X.cpu().double(), Wt.cpu().double(), dY.cpu().double()
    ref = {"Y": F_.conv2d(x, w, stride=s, padding=p), "dX": F_.conv_transpose2d(d, w, stride=s, padding=p, output_padding=((H + 2 * p - F) % s, (W + 2 * p - F) % s))}
    for name, got, K in (("Y", Y, IC * F * F), ("dX", dX, OC * F * F)):
        y = ref[name].numpy()
        np.testing.assert_allclose(to_np(got), np.where(np.abs(y) > 3.4028235e38, np.copysign(np.inf, y), y), rtol=K * 2.0**-23, atol=K * 2.0**-20,
                                   equal_nan=True, err_msg=name)
    # the weight gradient of the channels that meet only numbers
    clean = [c for c in range(IC) if c not in (1, 3, IC - 1)]
    rows = [o for o in range(OC) if o not in (2, OC - 1)]
    xr, dr = x[:, clean], d[:, rows]
    wr = torch.zeros(len(rows), len(clean), F, F, dtype=torch.double, requires_grad=True)
    F_.conv2d(xr, wr, stride=s, padding=p).backward(dr)
    got = dW.cpu().double()[rows][:, clean]
    assert (got - wr.grad).norm() <= 2.0**-24 * (N * g.OH * g.OW) ** 0.5 * wr.grad.norm()
    assert not dW.cpu()[:, IC - 1].isfinite().any(dim=(1, 2)).all() and not dW.cpu()[2].isfinite().all()
