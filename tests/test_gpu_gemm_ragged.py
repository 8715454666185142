"""Products on either side of the lines from which split operands take them (csrc/crb_gemm.hip, split_pays_sooner): rows that are
no multiple of 16 bytes long from 3 * 2^24 multiply-adds, 2^27 where the contraction is cut; whole rows from 2^27 where it is not."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# (M, N, K)
SIZES = [(270, 1277, 150), (271, 1277, 145), (1201, 875, 64), (1201, 890, 63), (768, 912, 192), (768, 916, 191), (512, 513, 511), (513, 513, 512),
         (129, 2031, 513), (33, 2047, 1987)]


@pytest.mark.parametrize("size", SIZES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("form", ["nn", "nt", "tn", "nta"])
def test_products_around_the_lines(dev, form, size):
    import torch
    from crusaderbackend_amd import capi

    M, N, K = size
    A, B = torch.randn(M, K, device=dev), torch.randn(K, N, device=dev)
    a, b = A.t().contiguous() if form == "tn" else A, B.t().contiguous() if form in ("nt", "nta") else B
    C = torch.zeros(M, N, device=dev)
    getattr(capi, "sgemm_" + form)(a, b, C, M, N, K)
    ref = A.cpu().double() @ B.cpu().double()
    # every product and sum rounds once: 0.29 * 2^-23 of a partial sum each, 0.71 of the last one in the mean
    assert (C.cpu().double() - ref).norm() <= 2 * np.sqrt(K) * 2.0**-25 * ref.norm()


@pytest.mark.parametrize("batch,IN,OUT", [(179, 2715, 359), (150, 1277, 270), (64, 2049, 513)])
def test_dense_layers_around_the_lines(dev, batch, IN, OUT):
    """All three products of a layer, the bias and its gradient; with less scratch than slices take the same bits."""
    import torch
    from crusaderbackend_amd import capi

    X, W, b, dY = (torch.randn(*s, device=dev) for s in ((batch, IN), (OUT, IN), (OUT,), (batch, OUT)))
    dW0, dB0 = torch.randn(OUT, IN, device=dev), torch.randn(OUT, device=dev)

    def run(stream):
        Y, dX, dW, dB = torch.empty(batch, OUT, device=dev), torch.empty(batch, IN, device=dev), dW0.clone(), dB0.clone()
        torch.cuda.synchronize()
        capi.linear_fwd(X, W, b, Y, batch, IN, OUT, capi.CRB_FLAG_RELU, stream=stream)
        capi.linear_dgrad(dY, W, dX, batch, IN, OUT, stream=stream)
        capi.linear_wgrad(dY, X, dW, dB, batch, IN, OUT, stream=stream)
        torch.cuda.synchronize()
        return Y, dX, dW, dB

    got = run(torch.cuda.current_stream())
    x, w, d = (t.cpu().double() for t in (X, W, dY))
    ref = (x @ w.t() + b.cpu().double()).relu(), d @ w, dW0.cpu().double() + d.t() @ x, dB0.cpu().double() + d.sum(0)
    for g, r, K in zip(got, ref, (IN, OUT, batch, batch)):
        assert (g.cpu().double() - r).norm() <= 2 * np.sqrt(K + 2) * 2.0**-25 * r.norm()
    side = torch.cuda.Stream(device=dev)
    most = max(capi.gemm_workspace_bytes(*s, 1) for s in ((batch, OUT, IN), (batch, IN, OUT), (OUT, IN, batch)))
    if most < 1024:
        return
    little = torch.empty(most // 4 - 128, device=dev)
    try:
        capi.bind_workspace(little, stream=side)
        assert all(torch.equal(p, q) for p, q in zip(got, run(side)))
    except capi.CrbError as e:  # (where the fp32 engine would be refused too)
        assert e.status == capi.CRB_EWORKSPACE
    finally:
        capi.bind_workspace(None, stream=side)


# K one past / one short of a quad, of a wave's share and of the group of loads; blocks of 16 that are not full
@pytest.mark.parametrize("size", [(1, 1, 1), (17, 33, 3), (16, 16, 5), (5, 70, 66), (33, 31, 255), (20, 18, 257), (130, 125, 1021), (30, 510, 4090)],
                         ids=lambda s: "x".join(map(str, s)))
def test_small_products_on_ragged_contractions(dev, size):
    """Both operands contiguous along a contraction that is no multiple of four, at any address: the same bits."""
    import torch
    from crusaderbackend_amd import capi

    M, N, K = size

    def at(t, off):
        buf = torch.full((t.numel() + 8,), float("nan"), device=dev)
        buf[off:off + t.numel()] = t.flatten()
        return buf[off:off + t.numel()].view(t.shape)

    A, B, bias, C0 = torch.randn(M, K, device=dev), torch.randn(N, K, device=dev), torch.randn(N, device=dev), torch.randn(M, N, device=dev)
    first = None
    for oa, ob in ((0, 0), (1, 0), (3, 2)):
        Y, C = torch.empty(M, N, device=dev), C0.clone()
        capi.linear_fwd(at(A, oa), at(B, ob), bias, Y, M, K, N, capi.CRB_FLAG_RELU)
        capi.sgemm_nta(at(A, oa), at(B, ob), C, M, N, K, 1)
        first = first or (Y, C)
        assert torch.equal(Y, first[0]) and torch.equal(C, first[1])
    p = A.cpu().double() @ B.cpu().double().t()
    for got, ref in ((first[0], (p + bias.cpu().double()).relu()), (first[1], p + C0.cpu().double())):
        assert (got.cpu().double() - ref).norm() <= 2 * np.sqrt(K + 2) * 2.0**-25 * (p.norm() + ref.norm())


@pytest.mark.parametrize("K", [3, 8, 30])
def test_small_products_over_a_batch(dev, K):
    """Entries that end inside a quad, and whole ones at an odd address."""
    import torch
    from crusaderbackend_amd import capi

    M, N, batch = 19, 33, 7
    A, B = (torch.randn(batch * r * K + 1, device=dev)[1:].view(batch, r, K) for r in (M, N))
    C = torch.zeros(M, N, device=dev)
    capi.sgemm_nta(A, B, C, M, N, K, batch)
    ref = sum(a.double() @ b.double().t() for a, b in zip(A.cpu(), B.cpu()))
    assert (C.cpu().double() - ref).norm() <= 2 * np.sqrt(K * batch) * 2.0**-25 * ref.norm()
