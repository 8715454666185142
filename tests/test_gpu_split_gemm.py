"""Products on the split engine (three bf16 parts per float, csrc/igemm_split.h) where its tiles and slabs end: remainders of
every tile edge and of the K slabs, operands off the 16-byte grid, cut contractions, accumulation, row sums; and the
claim that nothing of the operands' 24 bits is lost."""
import numpy as np
import pytest

from oracle import seblas_oracle as orc
from tests.util import assert_close, to_dev, to_np, uniform

pytestmark = pytest.mark.gpu

# (M, N, K), at least 2^28 multiply-adds: one past / one short of the 256, 128 and 64 tiles, K one past / one short of slabs of
# 16, 32 and 64, a contraction of a single ragged slab, tall and flat results, few tiles under a long (cut) contraction
SIZES = [(1025, 1023, 257), (4097, 4095, 17), (129, 2047, 1025), (65, 4097, 1031), (8191, 63, 543), (256, 1024, 1025), (97, 101, 27409),
         (515, 514, 1033), (2048, 2049, 64)]


def product(capi, form, A, B, C, M, N, K):
    getattr(capi, "sgemm_" + form)(A, B, C, M, N, K)


@pytest.mark.parametrize("form", ["nn", "nt", "tn", "nta"])
@pytest.mark.parametrize("size", SIZES, ids=lambda s: "x".join(map(str, s)))
def test_split_product_edges(dev, form, size):
    import torch
    from crusaderbackend_amd import capi

    M, N, K = size
    A, B = uniform(M + K, M, K), uniform(N + K, K, N)
    ref = orc.sgemm(A, B)
    a = np.ascontiguousarray(A.T) if form == "tn" else A
    b = np.ascontiguousarray(B.T) if form in ("nt", "nta") else B

    def off_grid(x):  # 4 bytes past a 16-byte boundary
        buf = torch.empty(x.size + 1, device=dev)
        buf[1:].copy_(torch.from_numpy(x.reshape(-1)))
        return buf[1:]

    C0 = uniform(7, M, N) if form == "nta" else np.zeros((M, N), np.float32)  # nta accumulates
    C = to_dev(C0, dev)
    product(capi, form, off_grid(a), off_grid(b), C, M, N, K)
    torch.cuda.synchronize()
    assert_close(to_np(C), ref + C0, K, f"{form} {size}")


@pytest.mark.parametrize("batch,IN,OUT", [(257, 1025, 1031), (1031, 513, 519)])
def test_split_dense_layer_gradients(dev, batch, IN, OUT):
    import torch
    from crusaderbackend_amd import capi

    dY, X = uniform(1, batch, OUT), uniform(2, batch, IN)
    dW0, dB0 = uniform(3, OUT, IN), uniform(4, OUT)
    dW, dB = to_dev(dW0, dev), to_dev(dB0, dev)
    capi.linear_wgrad(to_dev(dY, dev), to_dev(X, dev), dW, dB, batch, IN, OUT)
    torch.cuda.synchronize()
    assert_close(to_np(dW), dW0 + dY.astype(np.float64).T @ X, batch, "dW")
    assert_close(to_np(dB), dB0 + dY.astype(np.float64).sum(0), batch, "dB")


def test_split_product_loses_nothing_of_its_operands(dev):
    """Exact results where fp32 has them: operands of 24 significant bits times powers of two, one product per result (a
    permutation), come back bit for bit; and the distance of a long sum from float64 stays under that of a sum whose every
    product and addition rounds once to fp32, sqrt(K) * 2^-24 in the 2-norm for operands of one scale."""
    import torch
    from crusaderbackend_amd import capi

    n = 1024
    A = uniform(5, n, n)
    perm = np.random.RandomState(6).permutation(n)
    B = np.zeros((n, n), np.float32)
    B[perm, np.arange(n)] = np.ldexp(1.0, np.arange(n) % 9 - 4).astype(np.float32)
    C = torch.empty(n, n, device=dev)
    capi.sgemm_nn(to_dev(A, dev), to_dev(B, dev), C, n, n, n)
    torch.cuda.synchronize()
    assert np.array_equal(to_np(C), A[:, perm] * B[perm, np.arange(n)])

    B = uniform(8, n, n)
    capi.sgemm_nn(to_dev(A, dev), to_dev(B, dev), C, n, n, n)
    torch.cuda.synchronize()
    exact = A.astype(np.float64) @ B
    assert np.linalg.norm(to_np(C) - exact) <= np.sqrt(n) * 2.0**-24 * np.linalg.norm(exact)


# 256 x 256, 128 x 128 and 64 x 64 tiles, a cut contraction
@pytest.mark.parametrize("size", [(4096, 4095, 32), (2048, 2048, 65), (1024, 1024, 257), (256, 1024, 1025)], ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("form", ["nn", "nt", "tn", "wgrad"])
def test_infinities_and_the_largest_floats(dev, form, size):
    """Infinite operands and ones that round to infinity in 16 bits give what a product in fp32 gives: infinities of the right
    sign, NaN only where infinities meet or a NaN enters, finite results elsewhere."""
    import torch
    from crusaderbackend_amd import capi

    M, N, K = size
    A, B = uniform(1, M, K) / 2, uniform(2, K, N) / 2
    A[A == 0], B[B == 0] = 0.25, 0.25
    A[3, 5], A[M - 1, K - 1], A[40, 7] = np.inf, np.nan, 3.4e38
    B[2, 9], B[5, N - 1], B[K - 1, 70] = -np.inf, np.inf, -3.4e38
    A[65, 2], A[66, 2] = 0.5, -0.5
    with np.errstate(invalid="ignore", over="ignore"):
        ref = (A.astype(np.float64) @ B.astype(np.float64)).astype(np.float32)
    a = np.ascontiguousarray(A.T) if form in ("tn", "wgrad") else A
    b = np.ascontiguousarray(B.T) if form == "nt" else B
    if form == "wgrad":  # accumulates, with the row sums of A on the side
        C, dB = torch.zeros(M, N, device=dev), torch.zeros(M, device=dev)
        capi.linear_wgrad(to_dev(a, dev), to_dev(b, dev), C, dB, K, N, M)
    else:
        C = torch.empty(M, N, device=dev)
        product(capi, form, to_dev(a, dev), to_dev(b, dev), C, M, N, K)
    torch.cuda.synchronize()
    # K terms under 1/4, or that and one of 1.7e38, each rounded once or twice
    np.testing.assert_allclose(to_np(C), ref, rtol=K * 2.0**-23, atol=K * K * 2.0**-25, equal_nan=True)


def test_small_operands_keep_their_bits(dev):
    """Parts of operands down to 2^-110 are bf16 numbers, subnormal ones among them."""
    import torch
    from crusaderbackend_amd import capi

    n = 1024
    A = np.ldexp(np.float32(1) + np.abs(uniform(5, n, n)), -109).astype(np.float32)
    C = torch.empty(n, n, device=dev)
    capi.sgemm_nn(to_dev(A, dev), to_dev(np.eye(n, dtype=np.float32), dev), C, n, n, n)
    torch.cuda.synchronize()
    assert np.array_equal(to_np(C), A)


# 256 x 256, 128 x 128, 64 x 64 tiles of eight and of four waves, a cut contraction
@pytest.mark.parametrize("size", [(2304, 2300, 90), (2048, 2048, 65), (1024, 1024, 257), (1003, 1505, 777), (256, 1024, 1025)],
                         ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("form", ["nn", "nt", "tn", "nta"])
def test_products_that_overflow_throughout(dev, form, size):
    """No sum is finite: infinities of the right sign, NaN in one row, in the order of the finite product's time."""
    import torch
    from crusaderbackend_amd import capi

    M, N, K = size
    A, B = torch.rand(M, K, device=dev) + 1, torch.rand(K, N, device=dev) + 1
    big = A * 1e25
    big[M // 2] *= -1
    big[M // 3, K // 2] = float("nan")
    ref = torch.full((M, N), float("inf"), device=dev)
    ref[M // 2], ref[M // 3] = float("-inf"), float("nan")
    C = torch.zeros(M, N, device=dev)

    def lay(x, turn):
        return x.t().contiguous() if turn else x

    def timed(a, b):
        a, b = lay(a, form == "tn"), lay(b, form in ("nt", "nta"))
        t = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
        product(capi, form, a, b, C, M, N, K)
        t[0].record()
        product(capi, form, a, b, C, M, N, K)
        t[1].record()
        torch.cuda.synchronize()
        return t[0].elapsed_time(t[1])

    finite = timed(A, B)
    over = timed(big, B * 1e20)
    assert torch.equal(C.isnan(), ref.isnan()) and torch.equal(C.nan_to_num(0, 1, -1), ref.nan_to_num(0, 1, -1))
    # fp32 matrix instructions on operands straight from memory; a sum at a time it was 40 to 300 times as long
    assert over < 25 * max(finite, 0.02), (over, finite)


@pytest.mark.parametrize("form", ["nn", "nt", "tn", "nta"])
@pytest.mark.parametrize("size", [(2304, 2300, 90), (2048, 2048, 65), (1024, 1024, 257), (1003, 1505, 777)], ids=lambda s: "x".join(map(str, s)))
def test_operands_down_to_the_smallest_normal_float(dev, form, size):
    """Operands of 2^-126 and a little more against ones of 2^60 and back: as close to float64 as ordinary ones."""
    import torch
    from crusaderbackend_amd import capi

    M, N, K = size
    for ea, eb in ((-126, 60), (60, -126), (-126, -10)):
        A, B = (np.ldexp(np.float32(1) + np.abs(uniform(5 + i, *s)), e).astype(np.float32) for i, (s, e) in enumerate((((M, K), ea), ((K, N), eb))))
        A[::3], B[:, ::3] = -A[::3], -B[:, ::3]
        exact = A.astype(np.float64) @ B.astype(np.float64)
        a = np.ascontiguousarray(A.T) if form == "tn" else A
        b = np.ascontiguousarray(B.T) if form in ("nt", "nta") else B
        C = torch.zeros(M, N, device=dev)
        product(capi, form, to_dev(a, dev), to_dev(b, dev), C, M, N, K)
        torch.cuda.synchronize()
        # every product and addition rounds once, or (results under 2^-126) to the step of the subnormal numbers
        assert np.linalg.norm(to_np(C) - exact) <= np.sqrt(K) * 2.0**-24 * np.linalg.norm(exact) + np.sqrt(M * N) * K * 2.0**-150


@pytest.mark.parametrize("form", ["nn", "nt", "tn", "nta"])
@pytest.mark.parametrize("size", [(2304, 2300, 90), (2048, 2048, 65), (1024, 1024, 257), (1003, 1505, 777)], ids=lambda s: "x".join(map(str, s)))
def test_sums_of_one_product(dev, form, size):
    """Rows of A that hold one nonzero element, operands of 24 significant bits: what is left of a product is at most 2^-24 of it,
    a unit in the last place of a float in [1, 2) two of that, and its last rounding half a unit: 1.5 units."""
    import torch
    from crusaderbackend_amd import capi

    M, N, K = size
    A, at = np.zeros((M, K), np.float32), np.random.RandomState(3).randint(0, K, M)
    value, B = 1 + np.abs(uniform(4, M)), 1 + np.abs(uniform(5, K, N))
    A[np.arange(M), at] = value
    exact = value.astype(np.float64)[:, None] * B.astype(np.float64)[at]
    a = np.ascontiguousarray(A.T) if form == "tn" else A
    b = np.ascontiguousarray(B.T) if form in ("nt", "nta") else B
    C = torch.zeros(M, N, device=dev)
    product(capi, form, to_dev(a, dev), to_dev(b, dev), C, M, N, K)
    torch.cuda.synchronize()
    ulps = np.abs(to_np(C) - exact) / np.ldexp(1.0, np.floor(np.log2(exact)).astype(int) - 23)
    assert ulps.max() <= 1.5, (ulps.max(), np.sqrt((ulps**2).mean()))


# contractions that only the split products cut: 3 slices of 256 x 256 tiles, 3 of 128 x 128, 3 of 64 x 64 tiles of four waves
@pytest.mark.parametrize("size", [(3748, 1095, 1087), (389, 2305, 775), (3542, 135, 1044)], ids=lambda s: "x".join(map(str, s)))
def test_products_that_no_scratch_can_be_had_for(dev, size):
    """Recorded on a fresh stream, where nothing may be allocated: the bits of the eager call, for every form and epilogue."""
    import torch
    from crusaderbackend_amd import capi

    M, N, K = size
    assert capi.gemm_workspace_bytes(M, N, K, 1) > 0
    A, At, B, Bt = (torch.randn(*s, device=dev) for s in ((M, K), (K, M), (K, N), (N, K)))
    b, dB0, C0 = torch.randn(N, device=dev), torch.randn(M, device=dev), torch.randn(M, N, device=dev)

    def calls(C, dB, s):
        capi.sgemm_nn(A, B, C[0], M, N, K, stream=s)
        capi.sgemm_tn(At, B, C[1], M, N, K, stream=s)
        capi.sgemm_nta(A, Bt, C[2], M, N, K, stream=s)
        capi.linear_fwd(A, Bt, b, C[3], M, K, N, capi.CRB_FLAG_RELU, stream=s)
        capi.linear_wgrad(At, B, C[4], dB, K, N, M, stream=s)

    want, dB = C0.repeat(5, 1, 1), dB0.clone()
    calls(want, dB, torch.cuda.current_stream())
    got, dBg = C0.repeat(5, 1, 1), dB0.clone()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=torch.cuda.Stream(device=dev)):
        calls(got, dBg, torch.cuda.current_stream())
    for _ in range(3):
        got.copy_(C0.expand(5, M, N)), dBg.copy_(dB0)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(got, want) and torch.equal(dBg, dB)


@pytest.mark.parametrize("size", [(1024, 1024, 1024), (1003, 1505, 777)], ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("form", ["nn", "nt", "tn"])
def test_small_tiles_round_a_sum_once_per_sixteen_terms(dev, form, size):
    """64 x 64 tiles. A rounding is at most half of 2^-23 of the sum so far, in the mean 0.29 of it; the sums so far are 0.71 of the
    last one in the mean: sqrt(roundings) * 2^-25 at most, the K groups a few more."""
    import torch
    from crusaderbackend_amd import capi

    M, N, K = size
    A, B = torch.randn(M, K, device=dev), torch.randn(K, N, device=dev)
    C = torch.empty(M, N, device=dev)
    product(capi, form, A.t().contiguous() if form == "tn" else A, B.t().contiguous() if form == "nt" else B, C, M, N, K)
    ref = A.cpu().double() @ B.cpu().double()
    assert (C.cpu().double() - ref).norm() <= np.sqrt(K / 16 + 16) * 2.0**-25 * ref.norm()
