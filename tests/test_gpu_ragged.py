"""GPU tests of the bf16 products at sizes that no tile divides: ragged token counts (M of the
forward and input-gradient products, K of the weight gradients), K tails, odd sizes and unaligned
operands.  Every operand is followed by NaNs in its buffer, so a read past its end shows.

Tolerances: fp32 results are fp32 sums of exact bf16 products, 1e-5 normwise at these lengths
(<= 3000 terms: sqrt(3000) * 2^-24 = 3.3e-6); bf16 results are rounded once more, 2^-8."""
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

BF = torch.bfloat16


@pytest.fixture(scope="module")
def gn(gpu):
    import gn_bwd
    gn_bwd.lib()
    return gn_bwd


def guarded(g, *shape, std=1.0, offset=0):
    """A bf16 tensor at element `offset` of a buffer whose other elements are NaN."""
    n = 1
    for s in shape:
        n *= s
    buf = torch.full((offset + n + 4096,), float("nan"), device="cuda:0", dtype=BF)
    buf[offset:offset + n] = (torch.randn(n, device="cuda:0", generator=g) * std).to(BF)
    return buf[offset:offset + n].view(*shape)


def err(a, ref):
    return float((a.double() - ref).abs().max() / ref.abs().max().clamp(min=1e-30))


def gen(seed):
    g = torch.Generator(device="cuda:0")
    g.manual_seed(seed)
    return g


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("M,N,K", [(1, 8, 8), (8, 8, 1), (37, 264, 136), (136, 72, 1003), (257, 384, 63),
                                   (1003, 768, 72), (768, 776, 1003), (33, 50, 77), (131, 1001, 129),
                                   # K split over a block's waves: rings not filled, filled, reused
                                   (32, 32, 64), (40, 40, 320), (72, 264, 2112), (200, 136, 2600)])
def test_gemm_any_size(gn, ta, tb, M, N, K):
    g = gen(M + N + K)
    A = guarded(g, *((K, M) if ta else (M, K)))
    B = guarded(g, *((N, K) if tb else (K, N)))
    ref = (A.double().t() if ta else A.double()) @ (B.double().t() if tb else B.double())
    assert err(gn.gemm(A, B, bool(ta), bool(tb), out_dtype=torch.float32), ref) < 1e-5
    assert err(gn.gemm(A, B, bool(ta), bool(tb), out_dtype=BF), ref) < 2.0 ** -8
    C = torch.ones(M, N, device="cuda:0")
    gn.gemm(A, B, bool(ta), bool(tb), C=C, accumulate=True)
    assert err(C, ref + 1) < 1e-5


@pytest.mark.parametrize("K0,K1", [(72, 1000), (128, 8), (1001, 64)])
def test_gemm_two_ragged_segments(gn, K0, K1):
    g = gen(K0)
    A0, B0, A1, B1 = (guarded(g, K0, 136), guarded(g, K0, 200), guarded(g, K1, 136), guarded(g, K1, 200))
    ref = A0.double().t() @ B0.double() + A1.double().t() @ B1.double()
    C = gn.gemm(A0, B0, True, False, A1=A1, B1=B1, out_dtype=torch.float32)
    assert err(C, ref) < 1e-5


@pytest.mark.parametrize("offset", [1, 4])
def test_gemm_unaligned_operands(gn, offset):
    g = gen(offset)
    A, B = guarded(g, 200, 136, offset=offset), guarded(g, 136, 264, offset=offset)
    ref = A.double() @ B.double()
    assert err(gn.gemm(A, B, out_dtype=torch.float32), ref) < 1e-5


@pytest.mark.parametrize("T", [1, 7, 63, 65, 1003, 2999])
def test_linear_ragged_tokens(gn, T):
    """Forward with bias, backward with bias sums and the split-K workspace."""
    N, K = 264, 384
    g = gen(T)
    X, W, b, dY = guarded(g, T, K), guarded(g, N, K, std=0.05), guarded(g, N), guarded(g, T, N, std=0.1)
    x, w, dy = X.double(), W.double(), dY.double()
    assert err(gn.linear_fwd(X, W, b), x @ w.t() + b.double()) < 2.0 ** -8
    for acc in (False, True):
        out = dict(dX=torch.ones(T, K, device="cuda:0", dtype=BF), dW=torch.ones(N, K, device="cuda:0"),
                   db=torch.ones(N, device="cuda:0"))
        dX, dW, db = gn.linear_bwd(dY, X, W, accumulate=acc, **out)
        one = 1.0 if acc else 0.0
        assert err(dX, dy @ w + one) < 2.0 ** -8
        assert err(dW, dy.t() @ x + one) < 1e-5
        assert err(db, dy.sum(0) + one) < 1e-5


@pytest.mark.parametrize("T,d,H", [(1, 64, 136), (1003, 768, 1024), (130, 72, 200)])
def test_ffn_ragged_tokens(gn, T, d, H):
    """The fused down-projection + GLU gradients and the projections' backward from them."""
    g = gen(T + H)
    dY, Wd, act = guarded(g, T, d, std=0.1), guarded(g, d, H, std=0.05), guarded(g, T, H)
    gate, up, n = guarded(g, T, H), guarded(g, T, H), guarded(g, T, d)
    Wg, Wu = guarded(g, H, d, std=0.05), guarded(g, H, d, std=0.05)
    gu, dWd, dbd = gn.ffn_down_glu_bwd("reglu_up", dY, act, Wd, gate, up, need_db=True, ws=None)
    dA = dY.double() @ Wd.double()
    rg = torch.cat((dA * up.double().clamp(min=0), dA * gate.double() * (up.double() > 0)), 1)
    assert err(gu, rg) < 2.0 ** -8
    assert err(dWd, dY.double().t() @ act.double()) < 1e-5
    assert err(dbd, dY.double().sum(0)) < 1e-5
    dX, dWg, dWu, dbg, dbu = gn.glu_proj_bwd(gu, n, Wg, Wu, need_db=True, ws=None)
    G, U = gu.double()[:, :H], gu.double()[:, H:]
    assert err(dX, G @ Wg.double() + U @ Wu.double()) < 2.0 ** -8
    for got, ref in ((dWg, G.t() @ n.double()), (dWu, U.t() @ n.double()), (dbg, G.sum(0)), (dbu, U.sum(0))):
        assert err(got, ref) < 1e-5


def guarded32(g, *shape, offset=0):
    """As guarded, fp32."""
    n = 1
    for s in shape:
        n *= s
    buf = torch.full((offset + n + 4096,), float("nan"), device="cuda:0")
    buf[offset:offset + n] = torch.randn(n, device="cuda:0", generator=g)
    return buf[offset:offset + n].view(*shape)


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("M,N,K", [(1, 1, 129), (33, 31, 161), (64, 256, 784), (64, 10, 256), (163, 88, 1182),
                                   (6, 163, 1182), (1055, 1023, 300), (30, 50, 2000), (5, 7, 300),
                                   (36, 68, 140)])
@pytest.mark.parametrize("offset", [0, 1])
def test_gemm_fp32_any_size(gn, ta, tb, M, N, K, offset):
    """fp32 products off the six-product split's sizes on both tile sizes, few tiles of the split,
    K tails and unaligned operands; element-wise against K roundings of the sum of magnitudes."""
    g = gen(M + N + K)
    A = guarded32(g, *((K, M) if ta else (M, K)), offset=offset)
    B = guarded32(g, *((N, K) if tb else (K, N)), offset=offset)
    a, b = (A.double().t() if ta else A.double()), (B.double().t() if tb else B.double())
    ref, mag = a @ b, a.abs() @ b.abs()
    bound = 2.0 ** -24 * (K + 8)
    C = gn.gemm(A, B, bool(ta), bool(tb))
    assert bool(((C.double() - ref).abs() <= bound * mag).all())
    C = torch.ones(M, N, device="cuda:0")
    gn.gemm(A, B, bool(ta), bool(tb), C=C, accumulate=True)
    assert bool(((C.double() - ref - 1).abs() <= bound * (mag + 1)).all())


def test_gemm_fp32_in_order_of_k(gn):
    """Odd sizes add their products in increasing k with one rounding each: the result of a chain
    of fused multiply-adds, on 16 x 16 and 32 x 32 tiles alike."""
    g = gen(3)
    for M, N, K in ((17, 19, 131), (1001, 603, 131)):
        A, B = guarded32(g, M, K), guarded32(g, K, N)
        C = gn.gemm(A, B)
        ref = torch.zeros(M, N, device="cuda:0", dtype=torch.float64)
        for k in range(K):  # the fp64 product of two fp32 values is exact
            ref = (ref + A[:, k:k + 1].double() * B[k:k + 1].double()).float().double()
        # fp64 rounds the sum once more before fp32 does: a tie it creates may fall the other way
        assert float((C.double() != ref).float().mean()) < 1e-3
        assert err(C, ref) < 1e-6


def test_gemm_fp32_two_odd_segments_and_infinities(gn):
    g = gen(9)
    A0, B0, A1, B1 = (guarded32(g, 45, 301), guarded32(g, 301, 37), guarded32(g, 45, 9), guarded32(g, 9, 37))
    ref = A0.double() @ B0.double() + A1.double() @ B1.double()
    assert err(gn.gemm(A0, B0, A1=A1, B1=B1), ref) < 1e-5
    A0[3, 5] = float("inf")
    C = gn.gemm(A0, B0)
    assert bool(C[3].isinf().all()) and bool(C[[0, 1, 2, 4]].isfinite().all())


@pytest.mark.parametrize("M,N,K", [(9, 7, 130), (64, 256, 784), (200, 10, 333), (512, 4100, 256), (40, 12, 64)])
def test_linear_fwd_fp32_bias(gn, M, N, K):
    """The column bias in the epilogue of each fp32 kernel (matrix instruction, split, gemm_small)."""
    g = gen(M)
    X, W, b = guarded32(g, M, K), guarded32(g, N, K), guarded32(g, N)
    assert err(gn.linear_fwd(X, W, b), X.double() @ W.double().t() + b.double()) < 1e-5
    assert err(gn.linear_fwd(X, W), X.double() @ W.double().t()) < 1e-5
