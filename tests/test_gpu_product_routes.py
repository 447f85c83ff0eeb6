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
