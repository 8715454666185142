"""crb_conv_bwd where both gradients run on split operands: the slices' sum rides on the launch that splits the filters. The bits of the two calls."""
import pytest

from tests.util import launched

pytestmark = pytest.mark.gpu

# (N, IC, H, W, OC, F, stride, pad), how the slices are summed (rows of 16 bytes by 8 to 64 lanes, or as many single results from 1000 on): each way, filters in
# steps of 16 and 32 channels, K groups, residue classes
SHAPES = [(32, 64, 28, 28, 64, 3, 1, 1), (40, 64, 44, 40, 64, 3, 1, 1), (12, 64, 24, 24, 96, 3, 1, 1), (9, 41, 31, 33, 65, 3, 1, 1), (4, 256, 14, 14, 256, 3, 1, 1),
          (24, 30, 61, 47, 75, 5, 2, 2), (16, 64, 28, 28, 128, 3, 2, 1), (7, 64, 21, 19, 48, 5, 1, 2), (31, 24, 35, 24, 46, 3, 1, 1), (38, 26, 6, 20, 47, 3, 1, 1),
          (77, 25, 30, 55, 18, 3, 1, 1)]
LANES = [16, 16, 32, 1032, 64, 1032, 32, 32, 8, 1016, 1008]


def lanes(slices, count):
    if count % 4 == 0:
        return 8 if slices >= 64 else 16 if slices >= 32 else 32 if slices >= 16 or count < 1 << 17 else 64
    return 1032 if count >= 1 << 14 else 1016 if count >= 1 << 12 else 1008


@pytest.mark.parametrize("shape,way", zip(SHAPES, LANES), ids=lambda s: "x".join(map(str, s)) if isinstance(s, tuple) else str(s))
def test_the_two_calls(dev, shape, way):
    import torch
    from crusaderbackend_amd import capi

    N, IC, H, W, OC, F, s, p = shape
    g = capi.ConvGeom.make(N, IC, H, W, OC, F, F, s, s, p, p)
    X, Wt, dY, dW0 = (torch.randn(*a, device=dev) for a in ((N, IC, H, W), (OC, IC, F, F), (N, OC, g.OH, g.OW), (OC, IC, F, F)))
    need = capi.conv_wgrad_workspace_bytes(g)
    dX, dW = torch.empty_like(X), dW0.clone()
    capi.conv_dgrad(Wt, dY, dX, g)
    capi.conv_wgrad(dY, X, dW, g, workspace=torch.empty(need // 4 + 4, device=dev))
    torch.cuda.synchronize()

    def check(stream=None, workspace=None):
        a, b = torch.full_like(dX, 7.0), dW0.clone()
        torch.cuda.synchronize()
        capi.conv_bwd(Wt, dY, X, a, b, g, workspace=workspace, stream=stream)
        torch.cuda.synchronize()
        assert torch.equal(a, dX) and torch.equal(b, dW)

    ws = torch.empty(need // 4 + 4, device=dev)
    check(workspace=ws)
    check()
    assert lanes(need // (4 * dW.numel()), dW.numel()) == way
    a, b = torch.empty_like(dX), torch.empty_like(dW)
    kernels = [k for k, _ in launched(dev, lambda stream: capi.conv_bwd(Wt, dY, X, a, b, g, workspace=ws, stream=stream))]
    assert not any("splitk_reduce" in k for k in kernels), kernels
    assert any("filters_kernelILb1ELb1E" in k or "class_filters_kernelILb1E" in k for k in kernels), kernels
    side, shared = torch.cuda.Stream(device=dev), torch.empty((need + capi.conv_dgrad_workspace_bytes(g)) // 4 + 64, device=dev)
    try:
        capi.bind_workspace(shared, stream=side)  # split filters and slices in one place
        check(side, shared)
        capi.bind_workspace(shared[:64], stream=side)  # no room for split filters
        try:
            capi.conv_dgrad(Wt, dY, a, g, stream=side)
            alone = capi.CRB_OK
        except capi.CrbError as e:
            alone = e.status
        if alone == capi.CRB_OK:
            check(side, ws)
        else:  # the data gradient is refused alone, and so is the pair
            assert alone == capi.CRB_EWORKSPACE
            with pytest.raises(capi.CrbError) as e:
                check(side, ws)
            assert e.value.status == alone
    finally:
        capi.bind_workspace(None, stream=side)


@pytest.mark.parametrize("over,off", [("W", 0), ("W", 4), ("dY", 0), ("dY", 1), ("dX", 8), ("workspace", 0)])
@pytest.mark.parametrize("shape", [SHAPES[0], SHAPES[5]], ids=lambda s: "x".join(map(str, s)))
def test_weight_gradient_on_top_of_an_operand(dev, shape, over, off):
    """dW on the filters, on dY or on dX, and the filters on the workspace: what the two calls in their order leave there."""
    import torch
    from crusaderbackend_amd import capi

    N, IC, H, W, OC, F, s, p = shape
    g = capi.ConvGeom.make(N, IC, H, W, OC, F, F, s, s, p, p)
    n_w = OC * IC * F * F
    flat = {"X": N * IC * H * W, "W": n_w, "dY": N * OC * g.OH * g.OW, "dX": N * IC * H * W, "workspace": capi.conv_wgrad_workspace_bytes(g) // 4}
    start = {k: torch.randn(n + 16, device=dev) for k, n in flat.items()}
    start["dW"] = torch.randn(n_w, device=dev)

    def result(fn):
        t = {k: v.clone() for k, v in start.items()}
        if over == "workspace":
            t["W"] = t["workspace"][:n_w]
            t["W"].copy_(start["W"][:n_w])
        else:
            t["dW"] = t[over][off : off + n_w]
        torch.cuda.synchronize()
        fn(t)
        torch.cuda.synchronize()
        return [t[k] for k in ("dX", "dW", "dY")]

    def two(t):
        capi.conv_dgrad(t["W"], t["dY"], t["dX"], g)
        capi.conv_wgrad(t["dY"], t["X"], t["dW"], g, workspace=t["workspace"])

    for a, b in zip(result(two), result(lambda t: capi.conv_bwd(t["W"], t["dY"], t["X"], t["dX"], t["dW"], g, workspace=t["workspace"]))):
        assert torch.equal(a, b)
