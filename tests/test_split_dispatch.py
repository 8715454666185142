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


def test_few_images_stay_on_split_operands_where_these_are_ahead():
    """Long contractions into few channels over many pixels fill the small tiles of the few-image kernel several times over."""
    for shape in ((3, 608, 24, 16, 164, 3, 1, 1), (7, 752, 8, 8, 515, 3, 1, 1), (5, 656, 16, 8, 118, 3, 1, 1), (3, 752, 4, 32, 226, 3, 1, 1)):
        N, IC, H, W, OC = shape[:5]
        assert on_split_operands(queries(*shape)[0], shape), shape
    # VGG-16 on one image and on seven: slices of the result, or none
    for IC, H, OC in ((64, 16, 128), (128, 16, 128), (128, 8, 256), (256, 8, 256), (256, 4, 512), (512, 4, 512), (512, 2, 512)):
        for N in (1, 7):
            need = queries(N, IC, H, H, OC, 3, 1, 1)[0]
            assert need < 6 * IC * OC * 9 and need % (N * OC * H * H * 4) == 0


def test_pointwise_weight_gradients_ask_for_what_their_product_takes():
    """The accumulating NT form runs on split operands from 2^28 multiply-adds: under that, slices of the fp32 engine or none."""
    for shape, slices in (((8, 12939, 21, 21, 3, 1, 1, 0), 0), ((2, 3, 59, 59, 12064, 1, 1, 0), 0), ((82, 3, 12, 12, 4923, 1, 1, 0), 7)):
        assert queries(*shape)[2] == slices * shape[1] * shape[4] * 4


def test_wide_filter_weight_gradients_count_what_their_workgroups_add():
    """5x5, slices of the contraction: what a workgroup adds to the gradient counts beside its tiles, and the engine's estimate."""
    for shape, slices in (((2, 336, 5, 55, 295, 5, 2, 4), 2), ((28, 35, 35, 12, 482, 5, 2, 4), 18), ((10, 410, 23, 21, 32, 5, 2, 0), 4),  # on the engine
                          ((10, 410, 23, 21, 33, 5, 2, 0), 3), ((24, 30, 61, 47, 75, 5, 2, 2), 24),
                          ((5, 96, 15, 9, 319, 5, 1, 4), 3), ((11, 142, 6, 36, 162, 5, 1, 0), 3)):  # 64-wide blocks, not 32-wide ones uncut
        assert queries(*shape)[2] == slices * shape[1] * shape[4] * 100, shape


def test_strided_wide_filters_on_few_channels():
    """5x5 stride 2: long contractions into few channels over few pixels stay in the engine's slices; where split operands are taken no more
    channels are padded than the tile of 64 has."""
    for shape, slices in (((17, 286, 38, 5, 31, 5, 2, 1), 50), ((4, 382, 29, 5, 45, 5, 2, 2), 67), ((4, 481, 18, 3, 26, 5, 2, 4), 84), ((10, 410, 23, 21, 32, 5, 2, 0), 59)):
        N, IC, H, W, OC, F, s, p = shape
        assert queries(*shape)[0] == slices * N * OC * ((H + 2 * p - F) // 2 + 1) * ((W + 2 * p - F) // 2 + 1) * 4, shape
    assert queries(28, 146, 9, 6, 28, 5, 2, 4)[0] == (10 * 2 * 25 + 2) * 3072 + 28 * 28 * 7 * 5 * 4 * 10


def test_tilings_of_the_weight_gradient_beside_the_rows_kernel():
    """What a tile of the transposing kernel is charged against the rows kernel does not move the choice between its own two tilings, where the
    rows kernel is not for the layer: ten slices, not twenty-one of 64-wide blocks, three instead of seven, one instead of three."""
    for shape, slices in (((45, 96, 37, 8, 256, 3, 1, 1), 10), ((36, 96, 19, 32, 256, 3, 1, 1), 10), ((10, 64, 50, 32, 376, 3, 1, 1), 10), ((7, 469, 12, 8, 261, 3, 1, 1), 0),
                          ((83, 64, 44, 33, 64, 3, 1, 1), 61), ((55, 355, 7, 7, 189, 3, 1, 1), 3), ((22, 32, 50, 50, 192, 3, 1, 2), 39), ((64, 64, 15, 15, 320, 3, 1, 2), 12)):
        assert queries(*shape)[2] == slices * shape[1] * shape[4] * 36, shape


def test_rows_weight_gradients_stay_in_the_scratch_of_the_kernel_before():
    """What the transposing kernel takes without slices, or with no more of them than the built-in buffer holds, the rows kernel takes so too:
    crb_conv_wgrad_noalloc and calls without scratch are refused nothing."""
    for N, IC, H, W, OC in ((4, 199, 10, 10, 316), (5, 206, 9, 10, 87), (1, 85, 21, 22, 281), (5, 452, 10, 10, 40)):
        assert queries(N, IC, H, W, OC, 3, 1, 1)[2] == 0, (N, IC, H, W, OC)
    for N, IC, H, W, OC in ((51, 481, 18, 18, 32), (59, 128, 29, 30, 57), (4, 315, 60, 56, 32), (14, 255, 11, 14, 160), (27, 158, 10, 10, 155), (13, 64, 56, 56, 64)):
        assert 0 < queries(N, IC, H, W, OC, 3, 1, 1)[2] <= 8 << 20, (N, IC, H, W, OC)
