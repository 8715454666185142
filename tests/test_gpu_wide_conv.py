"""Convolutions on split operands, 32 channels a step (csrc/conv_split_wide.h), where tiles, chunks, strips and slices end."""
import numpy as np
import pytest

from tests.util import assert_close, he_normal, launched, normal, to_dev, to_np

pytestmark = pytest.mark.gpu

# (N, IC, H, W, OC, pad), pass, channels of a tile, slices, workgroups: channels one past and one short of 32 and 64, a last pixel tile of a few pixels, strips, a
# chunk of which half is padding, every padding of 3x3, tiles of 32, 64 and 128 channels, with slices (of one chunk, of several) and without
SHAPES = [((33, 20, 39, 41, 63, 1), "fwd", 64, 1, 423), ((17, 28, 44, 41, 229, 1), "fwd", 64, 1, 984), ((31, 128, 40, 39, 61, 1), "dgrad", 64, 1, 756),
          ((31, 61, 40, 39, 129, 1), "fwd", 32, 1, 945), ((41, 23, 54, 52, 32, 1), "fwd", 32, 1, 450), ((70, 64, 41, 37, 31, 0), "fwd", 32, 1, 384),
          ((70, 64, 41, 37, 31, 2), "dgrad", 64, 1, 853), ((40, 96, 29, 131, 40, 1), "fwd", 64, 1, 1206), ((300, 64, 13, 13, 60, 1), "dgrad", 64, 1, 397),
          ((62, 19, 5, 39, 225, 2), "fwd", 128, 1, 570), ((58, 196, 14, 21, 21, 0), "dgrad", 128, 1, 534), ((48, 181, 17, 25, 27, 1), "fwd", 64, 3, 498),
          ((47, 26, 11, 41, 189, 0), "dgrad", 64, 3, 510), ((66, 277, 7, 23, 103, 1), "fwd", 128, 3, 501), ((23, 255, 9, 26, 280, 0), "dgrad", 128, 3, 510),
          ((16, 279, 50, 5, 194, 2), "fwd", 32, 3, 483), ((49, 79, 38, 7, 284, 1), "dgrad", 32, 3, 459), ((15, 348, 18, 41, 26, 1), "fwd", 32, 11, 495)]

# the configuration's name by the channels of its tile, as the kernel's has it
CFG = {64: "ConvWideCfgILi2ELi2ELi256EEE", 128: "ConvWideCfgILi4ELi1ELi256EEE", 32: "ConvWideCfgILi1ELi4ELi384EEE"}


@pytest.mark.parametrize("shape,which,tile,slices,workgroups", SHAPES, ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else str(v))
def test_wide_steps(dev, shape, which, tile, slices, workgroups):
    """Against float64, with operands that are not finite, and with less scratch than the call takes: the same bits. The kernels are the ones meant."""
    import torch
    import torch.nn.functional as F_
    from crusaderbackend_amd import capi

    N, IC, H, W, OC, p = shape
    F = 3
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

    kernels = launched(dev, lambda stream: call(xd, out, stream=stream))
    assert [n for k, n in kernels if "conv_wide_kernel" in k and CFG[tile] + "Lb0E" in k] == [workgroups], kernels
    assert any("ordered_reduce_kernel" in k for k, _ in kernels) == (slices > 1)

    again, side, little = torch.empty_like(out), torch.cuda.Stream(device=dev), torch.empty(need // 4 - 256, device=dev)
    torch.cuda.synchronize()
    try:
        capi.bind_workspace(little, stream=side)
        call(xd, again, stream=side)
        side.synchronize()
        assert torch.equal(out, again)

        def without(stream):
            capi.bind_workspace(little, stream=stream)
            call(xd, again, stream=stream)
            capi.bind_workspace(None, stream=stream)

        kernels = launched(dev, without)  # (a launch a slice)
        assert [CFG[tile] + "Lb1E" in k for k, _ in kernels] == [True] * slices, kernels
    finally:
        capi.bind_workspace(None, stream=side)

    x[0, 1, -1, -1], x[N - 1, 3, 0, 0], x[N // 2, 5, 4, min(7, x.shape[3] - 1)] = float("inf"), -3.4e38, float("-inf")
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
