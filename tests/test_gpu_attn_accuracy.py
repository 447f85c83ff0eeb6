"""GPU test of the bf16 attention forward's precision on peaked rows: the leading weight of a row is
exactly 1 in bf16, whichever tile its key lies in and however little its score exceeds the earlier
tiles' maximum."""
import math

import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def gn(gpu):
    import gn_bwd
    gn_bwd.lib()
    return gn_bwd


@pytest.mark.parametrize("mask", [False, True])
@pytest.mark.parametrize("D", [64, 128])
def test_leading_weight_is_exact(gn, D, mask):
    """Two keys matter in a row: one in the first tile (score 0) and one in a later tile whose score is
    4 to 7.9 above it (base 2); the rest lie far below.  Against 64 bits, each row of O is compared
    along the exact row: c = O . Oref / Oref . Oref.
    A bf16 rounding is off by at most half an ulp, 2^-9 to 2^-8 of the value: 1.6e-3 rms.
    A leading weight of exactly 1 leaves in c - 1 the other weight's rounding (1.6e-3 of at most 2^-4:
    1e-4) and the D roundings of O, weighted by O^2: 1.6e-3 sqrt(3 / D) for a normal V, 3.5e-4 at
    D = 64.  Together 3.6e-4 rms; a rounded leading weight, the same for the whole row, adds its own
    1.6e-3.  The line is between the two."""
    B, H, S = 1, 2, 256
    g = torch.Generator(device="cuda:0")
    g.manual_seed(D)
    over = torch.linspace(4.0, 7.9, S, device="cuda:0")  # base-2 lead of the later key, by row
    Q = torch.zeros(B, H, S, D, device="cuda:0")
    Q[..., 0] = over * math.log(2.0)
    K = torch.zeros(B, H, S, D, device="cuda:0")
    K[..., 0] = -8.0
    K[:, :, 5, 0] = 0.0
    K[:, :, 200, 0] = 1.0
    V = torch.randn(B, H, S, D, device="cuda:0", generator=g)
    Q, K, V = (t.bfloat16().contiguous() for t in (Q, K, V))
    keep = torch.ones(B, S, device="cuda:0")
    keep[:, 70:80] = 0.0
    O, lse = gn.attn_fwd(Q, K, V, scale=1.0, causal=False, rope="none", mask=keep if mask else None)
    for h in range(H):
        sc = Q[0, h].double() @ K[0, h].double().t().contiguous()
        if mask:
            sc.masked_fill_(keep[0] < 0.5, -math.inf)
        ref = torch.softmax(sc, -1) @ V[0, h].double()
        c = (O[0, h].double() * ref).sum(-1) / (ref * ref).sum(-1) - 1
        assert float(c.pow(2).mean().sqrt()) < 6e-4
        assert float((lse[0, h].double() - torch.logsumexp(sc, -1)).abs().max()) < 1e-5
