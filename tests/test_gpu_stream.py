"""GPU tests of the bf16-output products on blocks that walk several tiles: one round and more of
either tile height, tiles cut by every edge, one k-tile per output tile, K tails, two K segments of
different pitches, and the bias and accumulating stores.  Operands sit in buffers of NaNs and C in
a buffer whose guard rows and columns must stay.

Tolerance: one bf16 rounding of an fp32 sum, 2^-8 of the largest element as an upper bound."""
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

from test_gpu_ragged import BF, err, gen, guarded  # noqa: E402


@pytest.fixture(scope="module")
def gn(gpu):
    import gn_bwd
    gn_bwd.lib()
    return gn_bwd


# (M, N): one round of 256-row tiles, three of 256 with edges, two and three rounds of 128-row
# tiles (the last two end inside the final round), a single short tile row
SHAPES = [(2600, 2312), (8200, 2056), (2600, 2056), (4104, 2312), (40, 34000)]


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("M,N", SHAPES)
@pytest.mark.parametrize("K", [8, 64, 200, 768])
def test_streamed_products(gn, ta, tb, M, N, K):
    m = M if ta else M - 1  # rows of a k-contiguous operand may be any count
    g = gen(M + N + K)
    A = guarded(g, *((K, m) if ta else (m, K)))
    B = guarded(g, *((N, K) if tb else (K, N)))
    ref = (A.double().t() if ta else A.double()) @ (B.double().t() if tb else B.double())
    buf = torch.full((m + 8, N), 7.0, device="cuda:0", dtype=BF)
    gn.gemm(A, B, bool(ta), bool(tb), C=buf[:m])
    assert err(buf[:m], ref) < 2.0 ** -8
    assert bool((buf[m:] == 7).all())
    C = torch.full((m, N), 2.0, device="cuda:0", dtype=BF)
    gn.gemm(A, B, bool(ta), bool(tb), C=C, accumulate=True)
    assert err(C, ref + 2) < 2.0 ** -8


@pytest.mark.parametrize("M,N,K", [(2600, 2312, 768), (8200, 2056, 72), (129, 34000, 136)])
def test_streamed_bias(gn, M, N, K):
    g = gen(K)
    x, w, b = guarded(g, M, K), guarded(g, N, K), guarded(g, N)
    ref = x.double() @ w.double().t() + b.double()
    assert err(gn.linear_fwd(x, w, b), ref) < 2.0 ** -8


@pytest.mark.parametrize("K0,K1", [(72, 200), (128, 8), (64, 64)])
def test_streamed_two_segments(gn, K0, K1):
    g = gen(K0 + K1)
    M, N = 4103, 2312
    A0, B0, A1, B1 = guarded(g, M, K0), guarded(g, K0, N), guarded(g, M, K1), guarded(g, K1, N)
    ref = A0.double() @ B0.double() + A1.double() @ B1.double()
    assert err(gn.gemm(A0, B0, A1=A1, B1=B1, out_dtype=BF), ref) < 2.0 ** -8


# fp32 weight gradients of more than two rounds of 256-row tiles (cut by both edges), K tails
@pytest.mark.parametrize("M,N,K", [(8200, 2056, 8), (8200, 2056, 200), (16392, 1032, 1003), (130, 131080, 64)])
def test_streamed_weight_gradient(gn, M, N, K):
    """|sum| error: fp32 accumulation of exact bf16 products, K 2^-24 of the largest term sum."""
    g = gen(M + K)
    A, B = guarded(g, K, M - M % 8), guarded(g, K, N)
    m = A.shape[1]
    ref = A.double().t() @ B.double()
    buf = torch.full((m + 8, N), 7.0, device="cuda:0")
    gn.gemm(A, B, True, False, C=buf[:m])
    tol = max(K, 64) * 2.0 ** -23
    assert err(buf[:m], ref) < tol
    assert bool((buf[m:] == 7).all())
    C = torch.full((m, N), 2.0, device="cuda:0")
    gn.gemm(A, B, True, False, C=C, accumulate=True)
    assert err(C, ref + 2) < tol


def test_streamed_weight_gradient_rows_split(gn):
    """[dWg; dWu] as one product: the second matrix begins inside a tile row."""
    g = gen(5)
    T, H, K = 203, 5000, 2056
    dO, gate, up, n = guarded(g, T, H), guarded(g, T, H), guarded(g, T, H), guarded(g, T, K)
    Wg, Wu = guarded(g, H, K), guarded(g, H, K)
    _, dWg, dWu, _, _ = gn.glu_linear_bwd("reglu_up", dO, gate, up, n, Wg, Wu)
    on = (up > 0).double()
    dg = (dO.double() * up.double() * on).to(BF).double()
    du = (dO.double() * gate.double() * on).to(BF).double()
    # the kernel forms each local gradient in fp32 and rounds once, as here: 2^-8 covers an
    # element that a double rounding moves
    assert err(dWg, dg.t() @ n.double()) < 2.0 ** -8
    assert err(dWu, du.t() @ n.double()) < 2.0 ** -8
