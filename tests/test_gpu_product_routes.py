"""GPU tests of the choice between the product kernels, at the sizes on either side of its lines,
against 64 bits on the same inputs.

Tolerances: fp32 results of bf16 operands are fp32 sums of exact products, sqrt(K) 2^-24 rms of the
result, < 2e-5 of its largest entry at every K here; bf16 results are rounded once more, 2^-8."""
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

BF = torch.bfloat16


@pytest.fixture(scope="module")
def gn(gpu):
    import gn_bwd
    gn_bwd.lib()
    return gn_bwd


def err(a, ref):
    return float((a.double() - ref).abs().max() / ref.abs().max().clamp(min=1e-30))


def rand(seed, *shape, dtype=BF, std=1.0):
    g = torch.Generator(device="cuda:0")
    g.manual_seed(seed)
    return (torch.randn(*shape, device="cuda:0", generator=g) * std).to(dtype)


@pytest.mark.parametrize("M,N,K", [(4096, 2048, 5632), (4100, 2048, 5640)])
def test_input_gradient_of_several_rounds_beside_its_weight_gradient(gn, M, N, K):
    """Large enough to fork without a graph; dX then takes a block per tile."""
    dY, X, W = rand(1, M, N, std=0.01), rand(2, M, K), rand(3, N, K, std=0.02)
    dX, dW, _ = gn.linear_bwd(dY, X, W, need_db=False)
    torch.cuda.synchronize()
    assert err(dX, dY.double() @ W.double()) < 2.0 ** -8
    assert err(dW, dY.double().t().contiguous() @ X.double()) < 2e-5


@pytest.mark.parametrize("K", [16384, 16392, 20008])
@pytest.mark.parametrize("M,N", [(16, 768), (65, 264), (300, 136)])
def test_few_rows_over_a_long_k(gn, M, N, K):
    """An LM head's dX on few tokens: K (the vocabulary) shared by a block's waves at any length."""
    A, B = rand(4, M, K), rand(5, K, N)
    assert err(gn.gemm(A, B, out_dtype=BF), A.double() @ B.double()) < 2.0 ** -8
    dW = gn.gemm(rand(6, K, 136), rand(7, K, 72), transA=True, out_dtype=torch.float32)
    assert err(dW, rand(6, K, 136).double().t().contiguous() @ rand(7, K, 72).double()) < 2e-5


@pytest.mark.parametrize("T", [1, 8, 63, 64, 65, 200, 1023, 1024, 1025])
@pytest.mark.parametrize("N,K", [(136, 72), (2056, 1040), (5640, 2056)])
@pytest.mark.parametrize("db", [False, True])
def test_weight_gradient_of_few_rows(gn, T, N, K, db):
    """Either side of 16 k-tiles (1024 rows), with ragged tiles, at one round of them and above, where
    the column sums of dY are taken apart; stored, then added to what is there."""
    dY, X, W = rand(8, T, N, std=0.01), rand(9, T, K), rand(10, N, K, std=0.02)
    ref, sums = dY.double().t().contiguous() @ X.double(), dY.double().sum(0)
    _, dW, dB = gn.linear_bwd(dY, X, W, need_dx=False, need_db=db)
    assert err(dW, ref) < 2e-5 and (not db or err(dB, sums) < 2e-5)
    gn.linear_bwd(dY, X, W, need_dx=False, need_db=db, dW=dW, db=dB, accumulate=True)
    assert err(dW, 2 * ref) < 2e-5 and (not db or err(dB, 2 * sums) < 2e-5)


def test_weight_gradient_of_few_rows_over_two_rounds_of_tiles(gn):
    dY, X = rand(11, 8, 8192), rand(12, 8, 4096)
    dW = gn.gemm(dY, X, transA=True, out_dtype=torch.float32)
    assert err(dW, dY.double().t().contiguous() @ X.double()) < 2e-5


@pytest.mark.parametrize("M,N,K", [
    (5, 33, 17), (64, 10, 32),                # scalar tiles
    (512, 10, 256), (70, 21, 300),            # MFMA chain, 16- and 32-wide
    (128, 256, 512), (130, 100, 264),         # 32 x 32 tiles of six products
    (2048, 1024, 1024), (2050, 1028, 1000),   # 128 x 128
    (64, 40000, 512), (33, 40004, 260)])      # 64 x 256
@pytest.mark.parametrize("shift", [0, 1])
def test_biased_fp32_forward_on_every_kernel(gn, M, N, K, shift):
    """The column bias added by the product's own kernel, aligned and not, and the product without it.
    fp32 sums: sqrt(K) 2^-24 rms of an entry, five times that over the largest of 2e6 entries, which is
    itself five times the rms: < 2e-6 of the largest at K <= 1024."""
    X, W = rand(13, M, K, dtype=torch.float32), rand(14, N, K, dtype=torch.float32)
    b = rand(15, N + 1, dtype=torch.float32)[shift:shift + N]
    ref = X.double() @ W.double().t()
    assert err(gn.linear_fwd(X, W), ref) < 2e-6
    assert err(gn.linear_fwd(X, W, b), ref + b.double()) < 2e-6


@pytest.mark.parametrize("M,N,K", [(1536, 1536, 16), (1540, 1532, 20), (768, 768, 16), (3072, 3072, 16),
                                   (1024, 1024, 64), (516, 772, 36)])
@pytest.mark.parametrize("tA,tB", [(False, True), (True, False)])
def test_fp32_product_of_short_k(gn, M, N, K, tA, tB):
    """Either side of the line between 32 x 32 and larger tiles, where K is a few 16-wide stages."""
    A = rand(16, *((K, M) if tA else (M, K)), dtype=torch.float32)
    B = rand(17, *((N, K) if tB else (K, N)), dtype=torch.float32)
    ref = (A.double().t() if tA else A.double()) @ (B.double().t() if tB else B.double())
    assert err(gn.gemm(A, B, transA=tA, transB=tB), ref) < 2e-6
