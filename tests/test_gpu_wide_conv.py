"""Convolutions on split operands, 32 channels a step (csrc/conv_split_wide.h), where tiles, chunks, strips and slices end."""
import numpy as np
import pytest

from tests.util import assert_close, he_normal, normal, to_dev, to_np

pytestmark = pytest.mark.gpu

# (N, IC, H, W, OC, F, pad), pass; 384 workgroups and more: channels one past and one short of 32 and 64, a last pixel tile of a few pixels, strips, a
# chunk of which half is padding, every padding of 3x3, tiles of 32, 64 and 128 channels
SHAPES = [((33, 20, 39, 41, 63, 3, 1), "fwd"), ((17, 28, 44, 41, 229, 3, 1), "fwd"), ((31, 128, 40, 39, 61, 3, 1), "dgrad"), ((31, 61, 40, 39, 129, 3, 1), "fwd"),
          ((41, 23, 54, 52, 32, 3, 1), "fwd"), ((70, 64, 41, 37, 31, 3, 0), "fwd"), ((70, 64, 41, 37, 31, 3, 2), "dgrad"), ((40, 96, 29, 131, 40, 3, 1), "fwd"),
          ((300, 64, 13, 13, 60, 3, 1), "dgrad"), ((41, 32, 52, 50, 30, 5, 2), "fwd")]


@pytest.mark.parametrize("shape,which", SHAPES, ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else v)
def test_wide_steps(dev, shape, which):
    """Against float64, with operands that are not finite, and with less scratch than the call takes: the same bits."""
    import torch
    import torch.nn.functional as F_
    from crusaderbackend_amd import capi

    N, IC, H, W, OC, F, p = shape
    g = capi.ConvGeom.make(N, IC, H, W, OC, F, F, 1, 1, p, p)
    fwd = which == "fwd"
    C_IN, C_OUT = (IC, OC) if fwd else (OC, IC)
    Wt, b = he_normal(2, OC, IC, F, F), normal(4, OC)
    x = torch.from_numpy(normal(1, N, IC, H, W) if fwd else normal(3, N, OC, g.OH, g.OW))
    out = torch.empty(*((N, OC, g.OH, g.OW) if fwd else (N, IC, H, W)), device=dev)
    need = capi.conv_fwd_workspace_bytes(g) if fwd else capi.conv_dgrad_workspace_bytes(g)
    assert need > 6 * F * F * C_IN * C_OUT  # (room for split filters)
    Wd, bd = to_dev(Wt, dev), to_dev(b, dev)

    def call(a, out, **kw):
        if fwd:
            capi.conv_fwd(Wd, a, out, bd, g, capi.CRB_FLAG_RELU, **kw)
        else:
            capi.conv_dgrad(Wd, a, out, g, **kw)

    def reference(a):
        w = torch.from_numpy(Wt).double()
        return (F_.conv2d(a.double(), w, torch.from_numpy(b).double(), padding=p).relu() if fwd else F_.conv_transpose2d(a.double(), w, padding=p)).numpy()

    xd = x.to(dev)
    call(xd, out)
    torch.cuda.synchronize()
    assert_close(to_np(out), reference(x), C_IN * F * F, f"{which} {shape}")

    again, side, little = torch.empty_like(out), torch.cuda.Stream(device=dev), torch.empty(need // 4 - 256, device=dev)
    torch.cuda.synchronize()
    try:
        capi.bind_workspace(little, stream=side)
        call(xd, again, stream=side)
        side.synchronize()
        assert torch.equal(out, again)
    finally:
        capi.bind_workspace(None, stream=side)

    x[0, 1, -1, -1], x[N - 1, 3, 0, 0], x[N // 2, 5, 4, 7] = float("inf"), -3.4e38, float("-inf")
    call(x.to(dev), out)
    torch.cuda.synchronize()
    ref = reference(x)
    with np.errstate(over="ignore"):
        ref32 = ref.astype(np.float32)
    got, plain = to_np(out), np.abs(ref) < 1e6
    assert np.array_equal(got[~np.isfinite(ref32)], ref32[~np.isfinite(ref32)], equal_nan=True)
    assert np.abs(got[plain] - ref[plain]).max() <= 1e-5 * np.sqrt(C_IN * F * F)
    big = np.isfinite(ref32) & ~plain  # one term of 3.4e38 beside small ones
    assert np.abs(got[big] / ref[big] - 1).max(initial=0) <= 1e-6
