"""Which calls the kernels on split operands take, seen from what the size queries say (no GPU is touched)."""
import pytest

from crusaderbackend_amd import capi


def queries(N, IC, H, W, OC, F, s, p):
    g = capi.ConvGeom.make(N, IC, H, W, OC, F, F, s, s, p, p)
    return capi.conv_fwd_workspace_bytes(g), capi.conv_dgrad_workspace_bytes(g), capi.conv_wgrad_workspace_bytes(g)


# the 3x3 layers of VGG-16 on CIFAR images, with the slices their fp32 weight gradients are cut into
@pytest.mark.parametrize("layer", [(64, 32, 64, 32), (64, 16, 128, 16), (128, 16, 128, 8), (128, 8, 256, 4), (256, 8, 256, 2), (256, 4, 512, 1),
                                   (512, 4, 512, 1)], ids=lambda s: "x".join(map(str, s)))
def test_width_grid_layers_train_on_the_fp32_kernels(layer):
    """A training step of these layers keeps its bits: none of its three passes runs on split operands (no room for split
    filters, slices of the fp32 weight gradient)."""
    IC, H, OC, slices = layer
    assert queries(128, IC, H, H, OC, 3, 1, 1) == (0, 0, slices * OC * IC * 36 if slices > 1 else 0)


def test_layers_of_the_built_in_buffer_stay_in_it():
    """Layers whose fp32 weight gradient takes slices of at most the built-in buffer's size, or none, need no more on split
    operands: crb_conv_wgrad_noalloc takes them, on the kernel that crb_conv_wgrad takes."""
    for (N, IC, H, W, OC, F, s, p), fp32 in (((8, 148, 24, 23, 210, 3, 2, 1), 5.34), ((12, 36, 51, 46, 165, 3, 2, 1), 5.92)):
        assert fp32 < queries(N, IC, H, W, OC, F, s, p)[2] / 2**20 <= 8, "on split operands"
    for shape in ((16, 739, 8, 7, 416, 3, 2, 1), (1, 544, 28, 27, 443, 3, 2, 1)):
        assert queries(*shape)[2] == 0


def test_short_weight_gradients_of_few_output_channels_stay_on_fp32():
    """Under 32 output channels and 400 MFLOP the fp32 slices (two per CU: twice as many) are the faster."""
    for shape, slices in (((2, 188, 27, 22, 28, 3, 1, 1), 5), ((51, 113, 7, 7, 26, 3, 1, 1), 10)):
        N, IC, H, W, OC, F, s, p = shape
        assert queries(*shape)[2] == slices * OC * IC * F * F * 4


def on_split_operands(query, shape):
    N, IC, H, W, OC, F, s, p = shape
    return 6 * OC * IC * F * F <= query < 8 * OC * IC * F * F + (64 << 20)


def test_wide_filters_are_split_where_that_pays():
    """A few small images against wide filters stay on fp32, in the little scratch of those kernels; larger work is split."""
    for shape in ((3, 1088, 4, 4, 1096, 5, 1, 2), (4, 1122, 5, 5, 1874, 5, 1, 2), (1, 1648, 10, 10, 2000, 3, 1, 1), (1, 1622, 11, 11, 679, 5, 1, 2),
                  (1, 4096, 7, 7, 4096, 3, 1, 1), (7, 1897, 7, 7, 1166, 3, 2, 1)):
        assert max(queries(*shape)[:2]) <= 64 << 20, shape
    for shape in ((6, 1143, 7, 7, 1163, 5, 1, 2), (3, 1335, 15, 15, 429, 3, 1, 1), (3, 869, 16, 17, 785, 3, 1, 1), (5, 1119, 7, 7, 436, 3, 1, 1)):
        assert all(on_split_operands(q, shape) for q in queries(*shape)[:2]), shape


def test_plans_are_kept_by_value():
    """A plan is formed once for a geometry, not on every call, and the places that plans are kept in do not mix them up."""
    import random
    import time

    rng = random.Random(1)
    shapes = []
    while len(shapes) < 600:
        F, s = rng.choice((3, 5)), rng.choice((1, 2))
        N, IC, H, W, OC = (int(2 ** rng.uniform(a, b)) for a, b in ((0, 6), (4, 8), (2.4, 6), (2.4, 6), (4, 8)))
        shapes.append((N, IC, H, W, OC, F, s, rng.randrange(F)))
    first = [queries(*x) for x in shapes]
    assert [queries(*x) for x in reversed(shapes)] == first[::-1]

    geoms = [capi.ConvGeom.make(32, 64, 56, 56, 64, 3, 3, 1, 1, 1, 1), capi.ConvGeom.make(16, 64, 28, 28, 64, 5, 5, 1, 1, 2, 2)]
    took = []
    for _ in range(5):
        t = time.perf_counter()
        for _ in range(500):
            for g in geoms:
                capi.conv_fwd_workspace_bytes(g), capi.conv_dgrad_workspace_bytes(g)
        took.append((time.perf_counter() - t) / 2000)
    assert min(took) < 3e-6, "5 to 8 us when formed anew"
