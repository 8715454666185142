"""Small products in one launch (csrc/gemm_tiny.h): ends of its groups of sixteen k, its waves and its blocks, and the products it takes from the engine."""
import numpy as np
import pytest

from tests.util import launched

pytestmark = pytest.mark.gpu

# (M, N, K): blocks that end early, single rows and columns, contractions of one to four groups a wave with 0 to 15 k behind them, waves without work,
# the last K of four and of eight waves, the most K, blocks and blocks * K that are taken and one more of each
SHAPES = [(1, 1, 1), (17, 15, 3), (1, 33, 64), (33, 1, 100), (16, 16, 16), (31, 65, 63), (128, 10, 512), (65, 200, 333), (100, 300, 640), (100, 300, 641), (50, 90, 1024),
          (50, 90, 1025), (12, 40, 2048), (128, 96, 352), (502, 15, 614), (41, 315, 818), (2304, 144, 16), (512, 1024, 18), (513, 1024, 18), (3, 272, 2049), (432, 256, 1024),
          (448, 256, 1025), (512, 512, 1024), (640, 256, 1024), (368, 784, 896)]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_small_products(dev, shape):
    """Three forms, with operands a word off a 16-byte address, beside a row of infinities and of NaN, which stay in their row."""
    import torch
    from crusaderbackend_amd import capi

    M, N, K = shape

    def at(t, off):
        return torch.empty(t.numel() + off, device=dev)[off:].view(t.shape).copy_(t)

    A, B = torch.randn(M, K), torch.randn(K, N)
    if M > 2:
        A[M - 1, K - 1], A[M // 2, 0] = float("inf"), float("nan")
    B[K - 1] = B[K - 1].abs() + 0.25
    ref = A.double() @ B.double()
    fine = torch.isfinite(ref)
    for form, a, b in (("nn", A, B), ("nt", A, B.t().contiguous()), ("tn", A.t().contiguous(), B)):
        for off in (0, 1):
            C = torch.full((M, N), 7.0, device=dev)
            getattr(capi, "sgemm_" + form)(at(a, off), at(b, off), C, M, N, K)
            got = C.cpu()
            assert (got[fine].double() - ref[fine]).norm() <= 2 * np.sqrt(K + 2) * 2.0**-25 * ref[fine].norm()
            assert torch.equal(got[~fine].isnan(), ref[~fine].isnan()) and bool((got[~fine & ref.isinf()] == float("inf")).all())


@pytest.mark.parametrize("batch,IN,OUT", [(128, 512, 10), (37, 700, 91), (16, 96, 352), (1, 1500, 33)])
def test_dense_layers(dev, batch, IN, OUT):
    """Bias, ReLU, both gradients added, and the bias gradient formed beside the weight gradient."""
    import torch
    from crusaderbackend_amd import capi

    X, W, b, dY = (torch.randn(*s, device=dev) for s in ((batch, IN), (OUT, IN), (OUT,), (batch, OUT)))
    dW0, dB0 = torch.randn(OUT, IN, device=dev), torch.randn(OUT, device=dev)
    Y, dX, dW, dB = torch.empty(batch, OUT, device=dev), torch.empty(batch, IN, device=dev), dW0.clone(), dB0.clone()
    capi.linear_fwd(X, W, b, Y, batch, IN, OUT, capi.CRB_FLAG_RELU)
    capi.linear_dgrad(dY, W, dX, batch, IN, OUT)
    capi.linear_wgrad(dY, X, dW, dB, batch, IN, OUT)
    x, w, d = (t.cpu().double() for t in (X, W, dY))
    ref = (x @ w.t() + b.cpu().double()).relu(), d @ w, dW0.cpu().double() + d.t() @ x, dB0.cpu().double() + d.sum(0)
    for g, r, K in zip((Y, dX, dW, dB), ref, (IN, OUT, batch, batch)):
        assert (g.cpu().double() - r).norm() <= 2 * np.sqrt(K + 2) * 2.0**-25 * r.norm()


# (form, M, N, K), taken from the engine or left to it: few rows of many columns, of which every XCD reads all, and the same where eight blocks or a multiple
# make a row of C; contractions of more than 1024 terms, shared by sixteen waves; few columns of many rows
LINES = [("nn", 103, 3732, 640, False), ("nn", 64, 2240, 1536, False), ("nn", 64, 1600, 1024, True), ("nn", 64, 2048, 1536, True), ("nn", 726, 188, 1812, False),
         ("nn", 368, 784, 896, True), ("nt", 1104, 64, 2016, False), ("nt", 118, 770, 1446, True), ("nt", 64, 1024, 1284, True), ("tn", 1536, 64, 1152, False), ("tn", 1536, 64, 704, True),
         ("tn", 45, 1373, 1608, False)]


@pytest.mark.parametrize("form,M,N,K,taken", LINES, ids=lambda v: str(v))
def test_products_taken_from_the_engine(dev, form, M, N, K, taken):
    import torch
    from crusaderbackend_amd import capi

    A, B, C = (torch.zeros(n, device=dev) for n in (M * K, N * K, M * N))
    names = [name for name, _ in launched(dev, lambda s: getattr(capi, "sgemm_" + form)(A, B, C, M, N, K, stream=s))]
    assert any("tiny_gemm_kernel" in n for n in names) == taken, names
