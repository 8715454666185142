"""Convolutions on the split engine (csrc/conv_split.h, conv_split_wgrad.h) where their tiles, strips, channel chunks and slices
end, against the CPU oracle."""
import numpy as np
import pytest

from oracle import seblas_oracle as orc
from tests.util import assert_close, he_normal, normal, to_dev, to_np

pytestmark = pytest.mark.gpu

# Edges of the layers, whichever kernels their sizes choose (PLANS below: a layer for every configuration of the split ones).
# (N, IC, H, W, OC, F, stride, pad): a last pixel tile of a few pixels, images narrower than a filter's reach and wider than a
# strip (uneven strips, a strip of padding columns), several images per tile, channels one past / one short of 16, 32 and 64,
# a contraction cut into slices, every padding, 5x5 with its rows in separate workgroups, stride 2 with odd extents
SHAPES = [(3, 64, 31, 33, 65, 3, 1, 1), (2, 33, 67, 61, 63, 3, 1, 1), (1, 47, 29, 131, 49, 3, 1, 1), (33, 96, 7, 5, 97, 3, 1, 1), (5, 129, 13, 14, 127, 3, 1, 0),
          (3, 80, 15, 17, 48, 3, 1, 2), (2, 300, 9, 11, 70, 3, 1, 1), (7, 31, 21, 19, 33, 5, 1, 2), (3, 40, 18, 23, 65, 5, 1, 0), (2, 36, 12, 50, 40, 5, 1, 4),
          # one image, one channel in the last chunk and tile: channels past it lie behind the tensor's end
          (1, 33, 67, 61, 65, 3, 1, 1), (1, 65, 61, 67, 129, 3, 2, 1), (1, 33, 37, 41, 65, 5, 1, 2),
          (4, 65, 33, 27, 97, 3, 2, 1), (3, 48, 30, 31, 66, 3, 2, 0), (70, 512, 4, 4, 96, 3, 1, 1), (64, 64, 32, 32, 64, 3, 1, 1), (9, 72, 20, 3, 80, 3, 1, 1),
          # under eight images on the width-specialised kernels' extents
          (1, 64, 32, 32, 64, 3, 1, 1), (2, 72, 16, 16, 128, 3, 1, 1), (3, 128, 8, 8, 80, 3, 1, 1), (7, 512, 4, 4, 512, 3, 1, 1)]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_split_convolution_edges(dev, shape):
    import torch
    from crusaderbackend_amd import capi

    N, IC, H, W, OC, F, s, p = shape
    g = capi.ConvGeom.make(N, IC, H, W, OC, F, F, s, s, p, p)
    X, Wt, dY, b = normal(1, N, IC, H, W), he_normal(2, OC, IC, F, F), normal(3, N, OC, g.OH, g.OW), normal(4, OC)
    dW0 = he_normal(5, OC, IC, F, F)
    Xd, Wd, dYd, bd, dW = (to_dev(a, dev) for a in (X, Wt, dY, b, dW0))
    Y, dX = torch.empty(N, OC, g.OH, g.OW, device=dev), torch.empty(N, IC, H, W, device=dev)
    capi.conv_fwd(Wd, Xd, Y, bd, g, capi.CRB_FLAG_RELU)
    capi.conv_dgrad(Wd, dYd, dX, g)
    capi.conv_wgrad(dYd, Xd, dW, g)
    torch.cuda.synchronize()
    assert_close(to_np(Y), np.maximum(orc.conv(Wt, X, b, s, s, p, p), 0), IC * F * F, f"forward {shape}")
    assert_close(to_np(dX), orc.convDerive(Wt, dY, (H, W), s, s, p, p), OC * F * F, f"data gradient {shape}")
    assert_close(to_np(dW), orc.convError(dY, X, dW0, s, s, p, p), N * g.OH * g.OW, f"weight gradient {shape}")
    dX2, dW2 = torch.empty_like(dX), to_dev(dW0, dev)
    capi.conv_bwd(Wd, dYd, Xd, dX2, dW2, g)
    torch.cuda.synchronize()
    assert torch.equal(dX, dX2) and torch.equal(dW, dW2)  # one call for both gradients: the same bits


@pytest.mark.parametrize("shape", [(32, 64, 28, 28, 64, 3, 1, 1), (32, 64, 28, 28, 64, 5, 1, 2)], ids=lambda s: "x".join(map(str, s)))
def test_layers_run_where_the_split_kernels_have_no_scratch(dev, shape):
    """A bound workspace too small for the split filters leaves the passes to the kernels that need none."""
    import torch
    from crusaderbackend_amd import capi

    N, IC, H, W, OC, F, s, p = shape
    g = capi.ConvGeom.make(N, IC, H, W, OC, F, F, s, s, p, p)
    assert capi.conv_fwd_workspace_bytes(g) > 256 and capi.conv_dgrad_workspace_bytes(g) > 256
    X, Wt, dY = normal(1, N, IC, H, W), he_normal(2, OC, IC, F, F), normal(3, N, OC, g.OH, g.OW)
    Xd, Wd, dYd = (to_dev(a, dev) for a in (X, Wt, dY))
    Y, dX = torch.empty(N, OC, g.OH, g.OW, device=dev), torch.empty(N, IC, H, W, device=dev)
    st, tiny = torch.cuda.Stream(device=dev), torch.empty(64, device=dev)
    torch.cuda.synchronize()
    try:
        capi.bind_workspace(tiny, stream=st)
        capi.conv_fwd(Wd, Xd, Y, None, g, stream=st)
        capi.conv_dgrad(Wd, dYd, dX, g, stream=st)
        st.synchronize()
    finally:
        capi.bind_workspace(None, stream=st)
    assert_close(to_np(Y), orc.conv(Wt, X, None, s, s, p, p), IC * F * F, f"forward {shape}")
    assert_close(to_np(dX), orc.convDerive(Wt, dY, (H, W), s, s, p, p), OC * F * F, f"data gradient {shape}")


@pytest.mark.parametrize("shape", [(3, 64, 31, 33, 65, 3, 1, 1), (2, 300, 9, 11, 70, 3, 1, 1), (7, 31, 21, 19, 33, 5, 1, 2), (4, 65, 33, 27, 97, 3, 2, 1)],
                         ids=lambda s: "x".join(map(str, s)))
def test_infinities_and_the_largest_floats(dev, shape):
    """Infinite operands and ones that round to infinity in 16 bits give what a contraction in fp32 gives: infinities of the
    right sign, NaN only where infinities meet or a NaN enters, finite results elsewhere."""
    import torch
    import torch.nn.functional as F_
    from crusaderbackend_amd import capi

    N, IC, H, W, OC, F, s, p = shape
    g = capi.ConvGeom.make(N, IC, H, W, OC, F, F, s, s, p, p)
    gen = torch.Generator().manual_seed(9)

    def half(*size):  # in [-0.5, 0.5], no zeros
        t = torch.rand(*size, generator=gen) - 0.5
        return torch.where(t == 0, torch.full_like(t, 0.25), t)

    X, Wt, dY = half(N, IC, H, W), half(OC, IC, F, F), half(N, OC, g.OH, g.OW)
    X[0, 3, 4, 5], X[N - 1, IC - 1, 3, 6], X[1, 1, 5, 4] = float("inf"), float("nan"), -3.4e38
    dY[0, 2, 2, 3], dY[N - 1, OC - 1, 2, 2] = float("-inf"), 3.4e38
    Xr, Wr = X.double().requires_grad_(), Wt.double().requires_grad_()
    Yr = F_.conv2d(Xr, Wr, stride=s, padding=p)
    Yr.backward(dY.double())
    Y, dX, dW = torch.empty(N, OC, g.OH, g.OW, device=dev), torch.empty(N, IC, H, W, device=dev), torch.zeros(OC, IC, F, F, device=dev)
    capi.conv_fwd(Wt.to(dev), X.to(dev), Y, None, g)
    capi.conv_dgrad(Wt.to(dev), dY.to(dev), dX, g)
    capi.conv_wgrad(dY.to(dev), X.to(dev), dW, g)
    torch.cuda.synchronize()
    for what, got, ref, K in (("Y", Y, Yr, IC * F * F), ("dX", dX, Xr.grad, OC * F * F), ("dW", dW, Wr.grad, N * g.OH * g.OW)):
        # K terms under 1/4, or that and one of 1.7e38, each rounded once or twice
        np.testing.assert_allclose(to_np(got), ref.detach().float().numpy(), rtol=K * 2.0**-23, atol=K * K * 2.0**-25, equal_nan=True, err_msg=what)


@pytest.mark.parametrize("shape", [(3, 64, 31, 33, 65, 3, 1, 1), (2, 300, 9, 11, 70, 3, 1, 1), (7, 31, 21, 19, 33, 5, 1, 2), (4, 65, 33, 27, 97, 3, 2, 1)],
                         ids=lambda s: "x".join(map(str, s)))
def test_layers_that_overflow_throughout(dev, shape):
    """Every product of a channel over- or underflows the largest float: infinities of the right sign, and ReLU keeps the positive."""
    import torch
    from crusaderbackend_amd import capi

    N, IC, H, W, OC, F, s, p = shape
    g = capi.ConvGeom.make(N, IC, H, W, OC, F, F, s, s, p, p)
    gen = torch.Generator().manual_seed(10)
    X, Wt = torch.rand(N, IC, H, W, generator=gen) + 1, torch.rand(OC, IC, F, F, generator=gen) + 1
    X, Wt = X * 1e25, Wt * 1e20
    Wt[OC // 2] *= -1
    ref = torch.full((N, OC, g.OH, g.OW), float("inf"))
    ref[:, OC // 2] = float("-inf")
    Y = torch.empty(N, OC, g.OH, g.OW, device=dev)
    for flags, want in ((0, ref), (capi.CRB_FLAG_RELU, ref.clamp(min=0))):
        capi.conv_fwd(Wt.to(dev), X.to(dev), Y, None, g, flags)
        torch.cuda.synchronize()
        assert torch.equal(Y.cpu(), want)


def check_against_float64(got, ref, K, what):
    """ref: float64 sums of K terms of one sign, of which each product and partial sum rounds to fp32 once (infinities: exactly)."""
    ref = ref.detach()
    np.testing.assert_allclose(to_np(got).astype(np.float64), np.where(np.abs(ref.numpy()) > 3.4028235e38, np.copysign(np.inf, ref.numpy()), ref.numpy()),
                               rtol=(K + 1) * 2.0**-23, equal_nan=True, err_msg=what)


# the last pixel of (17, 256, 7, 7) stands alone in its block of 32
LARGE = [(17, 256, 7, 7, 256, 3, 1, 1), (3, 64, 31, 33, 65, 3, 1, 1), (16, 64, 24, 23, 72, 5, 1, 2)]


@pytest.mark.parametrize("shape", LARGE, ids=lambda s: "x".join(map(str, s)))
def test_data_gradients_of_operands_that_round_to_infinity(dev, shape):
    """Output gradients beyond the largest bf16, one of them or all, with finite sums; and infinite ones throughout."""
    import torch
    import torch.nn.functional as F_
    from crusaderbackend_amd import capi

    N, IC, H, W, OC, F, s, p = shape
    g = capi.ConvGeom.make(N, IC, H, W, OC, F, F, s, s, p, p)
    assert capi.conv_dgrad_workspace_bytes(g) > OC * IC * F * F * 6  # the three parts of the filters: on split operands
    gen = torch.Generator().manual_seed(11)
    Wt, dY = torch.rand(OC, IC, F, F, generator=gen) * 0.5 + 0.25, torch.rand(N, OC, g.OH, g.OW, generator=gen) + 0.5
    one = dY.clone()
    one[N - 1, OC // 3, g.OH - 1, g.OW - 1] = 3.4e38
    negative = Wt.clone()
    negative[:, IC // 2] *= -1
    for what, w, dy in (("one", Wt, one), ("all", Wt * 1e-5, torch.full_like(dY, 3.4e38)), ("infinite", negative, torch.full_like(dY, float("inf")))):
        dX = torch.empty(N, IC, H, W, device=dev)
        capi.conv_dgrad(w.to(dev), dy.to(dev), dX, g)
        torch.cuda.synchronize()
        if what == "infinite":
            assert torch.equal(dX.cpu(), torch.where(torch.arange(IC).reshape(1, -1, 1, 1) == IC // 2, float("-inf"), float("inf")).expand_as(dX))
        else:
            ref = F_.conv_transpose2d(dy.double(), w.double(), stride=s, padding=p)
            check_against_float64(dX, ref, OC * F * F, what)


# 64 x 32 channels and 64 pixels a tile in one strip; 32 x 32 and 128; 5x5, whose filter rows are separate workgroups; stride 2
LARGE_W = [(17, 96, 13, 13, 64, 3, 1, 1), (3, 64, 31, 33, 65, 3, 1, 1), (16, 64, 24, 23, 72, 5, 1, 2), (4, 65, 33, 27, 97, 3, 2, 1)]


@pytest.mark.parametrize("shape", LARGE_W, ids=lambda s: "x".join(map(str, s)))
def test_weight_gradients_of_operands_that_round_to_infinity(dev, shape):
    """Inputs beyond the largest bf16 in five of a tile's 32 channels, or everywhere, with finite sums; and infinite gradients."""
    import torch
    from crusaderbackend_amd import capi

    N, IC, H, W, OC, F, s, p = shape
    g = capi.ConvGeom.make(N, IC, H, W, OC, F, F, s, s, p, p)
    gen = torch.Generator().manual_seed(12)
    X, dY = torch.rand(N, IC, H, W, generator=gen) + 0.5, torch.rand(N, OC, g.OH, g.OW, generator=gen) * 0.5 + 0.25
    few = X.clone()
    few[N - 1, 3:8, H // 2, W // 2] = 3.4e38
    infinite = dY.clone()
    infinite[:, OC // 2] = float("-inf")
    K = N * g.OH * g.OW
    for what, x, dy in (("few", few, dY), ("all", torch.full_like(X, 3.4e38), dY * (1 / K)), ("infinite", X, infinite)):
        dW = torch.zeros(OC, IC, F, F, device=dev)
        capi.conv_wgrad(dy.to(dev), x.to(dev), dW, g)
        torch.cuda.synchronize()
        ref = torch.nn.grad.conv2d_weight(torch.where(x.isinf(), 1.0, x).double(), (OC, IC, F, F), dy.double().nan_to_num(0, 0, 0), stride=s, padding=p)
        if what == "infinite":
            ref[OC // 2] = float("-inf")
        check_against_float64(dW, ref, K, what)


@pytest.mark.parametrize("shape", LARGE + LARGE_W[:1] + LARGE_W[3:], ids=lambda s: "x".join(map(str, s)))
def test_operands_down_to_the_smallest_normal_float(dev, shape):
    """Filters or activations of 2^-126 and a little more against ones of 2^60: as close to float64 as ordinary ones."""
    import torch
    import torch.nn.functional as F_
    from crusaderbackend_amd import capi

    N, IC, H, W, OC, F, s, p = shape
    g = capi.ConvGeom.make(N, IC, H, W, OC, F, F, s, s, p, p)
    gen = torch.Generator().manual_seed(13)

    def near(e, *size):
        t = torch.ldexp(torch.rand(*size, generator=gen) + 1, torch.tensor(e))
        return torch.where(torch.rand(*size, generator=gen) < 0.3, -t, t)

    for ew, ex in ((-126, 60), (60, -126)):
        Wt, X, dY = near(ew, OC, IC, F, F), near(ex, N, IC, H, W), near(ex, N, OC, g.OH, g.OW)
        Xs = near(186 + ex if ex < 0 else -126, N, IC, H, W)  # of the weight gradient: 2^60 against 2^-126 both ways
        Y, dX, dW = torch.empty(N, OC, g.OH, g.OW, device=dev), torch.empty(N, IC, H, W, device=dev), torch.zeros(OC, IC, F, F, device=dev)
        capi.conv_fwd(Wt.to(dev), X.to(dev), Y, None, g)
        capi.conv_dgrad(Wt.to(dev), dY.to(dev), dX, g)
        capi.conv_wgrad(dY.to(dev), Xs.to(dev), dW, g)
        torch.cuda.synchronize()
        Xr, Wr = torch.zeros(N, IC, H, W, dtype=torch.double, requires_grad=True), Wt.double()
        F_.conv2d(Xr, Wr, stride=s, padding=p).backward(dY.double())
        for what, got, ref, K in (("Y", Y, F_.conv2d(X.double(), Wr, stride=s, padding=p), IC * F * F), ("dX", dX, Xr.grad, OC * F * F),
                                  ("dW", dW, torch.nn.grad.conv2d_weight(Xs.double(), Wt.shape, dY.double(), stride=s, padding=p), N * g.OH * g.OW)):
            assert (got.cpu().double() - ref).norm() <= np.sqrt(K) * 2.0**-24 * ref.norm(), what


@pytest.mark.parametrize("shape", [(8, 148, 24, 23, 210, 3, 2, 1), (12, 36, 51, 46, 165, 3, 2, 1), (16, 739, 8, 7, 416, 3, 2, 1), (9, 48, 40, 41, 64, 3, 1, 1)],
                         ids=lambda s: "x".join(map(str, s)))
def test_the_gradient_that_allocates_nothing_has_the_same_bits(dev, shape):
    """crb_conv_wgrad on a workspace of the queried size, on the library's arena, on the built-in buffer, and recorded there."""
    import torch
    from crusaderbackend_amd import capi

    N, IC, H, W, OC, F, s, p = shape
    g = capi.ConvGeom.make(N, IC, H, W, OC, F, F, s, s, p, p)
    X, dY = torch.randn(N, IC, H, W, device=dev), torch.randn(N, OC, g.OH, g.OW, device=dev)
    need = capi.conv_wgrad_workspace_bytes(g)
    assert need <= capi.NOALLOC_SCRATCH_BYTES
    got = [torch.zeros(OC, IC, F, F, device=dev) for _ in range(4)]
    capi.conv_wgrad(dY, X, got[0], g, workspace=torch.empty(max(need, 4) // 4, device=dev))
    capi.conv_wgrad(dY, X, got[1], g)
    capi.conv_wgrad_noalloc(dY, X, got[2], g)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=torch.cuda.Stream(device=dev)):
        capi.conv_wgrad_noalloc(dY, X, got[3], g, stream=torch.cuda.current_stream())
    for _ in range(3):
        got[3].zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(got[0], x) for x in got[1:])
    if need:
        with pytest.raises(capi.CrbError) as ei:
            capi.conv_wgrad(dY, X, got[0], g, workspace=torch.empty(need // 8, device=dev))
        assert ei.value.status == capi.CRB_EWORKSPACE


# One layer for each kernel configuration, with and without a cut contraction: (N, IC, H, W, OC, F, stride, pad), pass,
# (configuration, slices)
PLANS = [((94, 78, 6, 7, 38, 3, 1, 0), "dgrad", (0, 1)), ((2, 31, 18, 10, 498, 3, 1, 1), "dgrad", (0, 11)), ((21, 333, 12, 3, 80, 3, 1, 0), "dgrad", (1, 1)),
         ((13, 206, 14, 3, 173, 3, 1, 0), "dgrad", (1, 4)), ((33, 129, 4, 5, 334, 3, 1, 0), "dgrad", (2, 11)), ((33, 129, 4, 14, 56, 3, 1, 0), "dgrad", (3, 1)),
         ((95, 37, 15, 3, 123, 3, 1, 0), "dgrad", (3, 2)), ((4, 28, 50, 20, 50, 3, 1, 1), "dgrad", (4, 1)), ((4, 24, 54, 7, 314, 3, 1, 0), "dgrad", (4, 7)),
         ((6, 35, 6, 38, 83, 3, 1, 2), "fwd", (0, 1)), ((2, 134, 10, 62, 27, 3, 1, 2), "fwd", (0, 3)), ((39, 72, 3, 34, 62, 3, 1, 0), "fwd", (1, 1)),
         ((2, 139, 5, 58, 119, 3, 1, 0), "fwd", (1, 3)), ((15, 399, 5, 28, 30, 3, 1, 0), "fwd", (2, 13)), ((73, 59, 15, 5, 36, 3, 1, 0), "fwd", (3, 1)),
         ((31, 402, 14, 3, 24, 3, 1, 1), "fwd", (3, 7)), ((3, 84, 35, 21, 30, 3, 1, 1), "fwd", (4, 1)), ((4, 116, 19, 40, 26, 3, 1, 1), "fwd", (4, 3)),
         ((6, 40, 58, 20, 80, 3, 2, 1), "fwd", (0, 1)), ((21, 150, 5, 4, 147, 3, 2, 2), "fwd", (0, 4)), ((7, 66, 6, 104, 118, 3, 2, 0), "fwd", (1, 1)),
         ((2, 496, 5, 15, 412, 3, 2, 0), "fwd", (1, 11)), ((10, 169, 53, 21, 25, 3, 2, 0), "fwd", (2, 6)), ((3, 29, 35, 29, 30, 5, 1, 0), "dgrad", (0, 1)),
         ((3, 75, 4, 108, 42, 5, 1, 1), "dgrad", (0, 3)), ((42, 24, 3, 60, 35, 5, 1, 1), "dgrad", (1, 1)), ((15, 85, 5, 12, 197, 5, 1, 0), "dgrad", (1, 13)),
         ((29, 171, 9, 5, 168, 5, 1, 0), "dgrad", (2, 6)), ((15, 138, 6, 37, 58, 5, 1, 0), "dgrad", (3, 1)), ((64, 18, 6, 8, 306, 5, 1, 0), "dgrad", (4, 15)),
         ((2, 24, 8, 112, 30, 5, 1, 4), "fwd", (0, 1)), ((2, 38, 11, 3, 405, 5, 1, 3), "fwd", (0, 3)), ((38, 16, 5, 7, 235, 5, 1, 1), "fwd", (1, 1)),
         ((43, 34, 16, 6, 57, 5, 1, 0), "fwd", (1, 3))]
# layers whose fp32 kernel would not run in less scratch either
REFUSED = {PLANS[i][0] for i in (3, 8, 10, 15, 16, 17, 20, 23, 26, 27, 28, 29, 30)}
# output channels of a tile, K groups, taps the filters run ahead
CONFIGURATIONS = ((64, 1, 4), (128, 1, 2), (128, 2, 2), (64, 4, 2), (32, 1, 4))


def plan_bytes(plan, C_IN, C_OUT, F, results):
    """Scratch of a plan: 3 KB of split filters per 32 output channels, 16 input channels and tap, in whole tiles and chunks."""
    OCT, KG, ahead = CONFIGURATIONS[plan[0]]
    filters = ((-(-C_OUT // OCT) * (OCT // 32)) * KG * -(-C_IN // (16 * KG)) * F * F + ahead) * 3072
    return -(-filters // 256) * 256 + (4 * plan[1] * results if plan[1] > 1 else 0)


@pytest.mark.parametrize("shape,which,plan", PLANS, ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else v)
def test_every_configuration(dev, shape, which, plan):
    """Against the oracle, with operands that are not finite against float64, and with less scratch than it takes: the same bits."""
    import torch
    import torch.nn.functional as F_
    from crusaderbackend_amd import capi

    N, IC, H, W, OC, F, s, p = shape
    g = capi.ConvGeom.make(N, IC, H, W, OC, F, F, s, s, p, p)
    X, Wt, dY, b = normal(1, N, IC, H, W), he_normal(2, OC, IC, F, F), normal(3, N, OC, g.OH, g.OW), normal(4, OC)
    fwd = which == "fwd"
    need = capi.conv_fwd_workspace_bytes(g) if fwd else capi.conv_dgrad_workspace_bytes(g)
    assert need == plan_bytes(plan, IC if fwd else OC, OC if fwd else IC, F, N * OC * g.OH * g.OW if fwd else N * IC * H * W)
    K = (IC if fwd else OC) * F * F
    Wd, bd = to_dev(Wt, dev), to_dev(b, dev)

    def call(x, out, **kw):
        if fwd:
            capi.conv_fwd(Wd, x, out, bd, g, capi.CRB_FLAG_RELU, **kw)
        else:
            capi.conv_dgrad(Wd, x, out, g, **kw)

    x = to_dev(X if fwd else dY, dev)
    out = torch.empty(*((N, OC, g.OH, g.OW) if fwd else (N, IC, H, W)), device=dev)
    call(x, out)
    torch.cuda.synchronize()
    ref = np.maximum(orc.conv(Wt, X, b, s, s, p, p), 0) if fwd else orc.convDerive(Wt, dY, (H, W), s, s, p, p)
    assert_close(to_np(out), ref, K, f"{which} {shape}")

    again, side, little = torch.empty_like(out), torch.cuda.Stream(device=dev), torch.empty(need // 4 - 64, device=dev)
    torch.cuda.synchronize()
    try:
        capi.bind_workspace(little, stream=side)
        call(x, again, stream=side)
        side.synchronize()
        assert torch.equal(out, again) and shape not in REFUSED
    except capi.CrbError as e:
        assert e.status == capi.CRB_EWORKSPACE and shape in REFUSED
    finally:
        capi.bind_workspace(None, stream=side)

    big = x.clone()
    big[0, 1, -1, -1], big[N - 1, 3, 0, 0] = float("inf"), -3.4e38
    call(big, out)
    torch.cuda.synchronize()
    y = (F_.conv2d(big.cpu().double(), torch.from_numpy(Wt).double(), torch.from_numpy(b).double(), stride=s, padding=p).relu() if fwd else
         F_.conv_transpose2d(big.cpu().double(), torch.from_numpy(Wt).double(), stride=s, padding=p)).numpy()
    # (where the one large operand is, it is all of the sum; beside it K terms of order 1, each rounded once or twice)
    np.testing.assert_allclose(to_np(out), np.where(np.abs(y) > 3.4028235e38, np.copysign(np.inf, y), y), rtol=K * 2.0**-23, atol=K * 2.0**-20, equal_nan=True)


@pytest.mark.parametrize("shape", [(8, 64, 56, 55, 64, 3, 1, 1), (17, 256, 13, 14, 256, 3, 1, 1), (4, 64, 28, 28, 64, 5, 1, 2), (4, 130, 57, 55, 97, 3, 2, 1)],
                         ids=lambda s: "x".join(map(str, s)))
def test_a_sum_is_rounded_once_per_sixteen_terms(dev, shape):
    """Activations behind a ReLU, half of them 0. A rounding is at most half of 2^-23 of the sum so far, in the mean 0.29 of it; the
    sums so far are 0.71 of the last one in the mean: sqrt(roundings) * 2^-25 at most, K groups and slices a few more. (The gradients
    too are of one sign: their weight gradient is nowhere near the cancellation that would make its error larger than that.)"""
    import torch
    import torch.nn.functional as F_
    from crusaderbackend_amd import capi

    N, IC, H, W, OC, F, s, p = shape
    g = capi.ConvGeom.make(N, IC, H, W, OC, F, F, s, s, p, p)
    gen = torch.Generator().manual_seed(21)
    X, Wt = torch.randn(N, IC, H, W, generator=gen).clamp(min=0), torch.randn(OC, IC, F, F, generator=gen)
    dY = torch.randn(N, OC, g.OH, g.OW, generator=gen).clamp(min=0)
    Y, dX = torch.empty(N, OC, g.OH, g.OW, device=dev), torch.empty(N, IC, H, W, device=dev)
    capi.conv_fwd(Wt.to(dev), X.to(dev), Y, None, g)
    ref = F_.conv2d(X.double(), Wt.double(), stride=s, padding=p)
    checks = [(Y, ref, IC * F * F)]
    if s == 1:
        capi.conv_dgrad(Wt.to(dev), dY.to(dev), dX, g)
        checks.append((dX, F_.conv_transpose2d(dY.double(), Wt.double(), stride=s, padding=p), OC * F * F))
    # (weight gradients: two roundings per sixteen pixels of a sum that K groups and slices hold in at least eight parts)
    dW = torch.zeros(OC, IC, F, F, device=dev)
    capi.conv_wgrad(dY.to(dev), X.to(dev), dW, g)
    checks.append((dW, torch.nn.grad.conv2d_weight(X.double(), Wt.shape, dY.double(), stride=s, padding=p), 2 * N * g.OH * g.OW / 8))
    torch.cuda.synchronize()
    for got, want, K in checks:
        assert (got.cpu().double() - want).norm() <= np.sqrt(K / 16 + 16) * 2.0**-25 * want.norm()
