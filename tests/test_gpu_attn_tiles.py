"""GPU tests of the bf16 attention kernels' tile selection: key masks that empty whole 64-key tiles
(which the kernels skip), windows of more than 64 tiles, ragged sequence ends, and maxima that
grow along a row (the forward rescales O on the tiles where some row's maximum moves).

Tolerance 2e-2 of the largest entry: bf16 probabilities and operands (2^-8), as the other bf16
attention tests."""
import math

import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

TOL = 2e-2


@pytest.fixture(scope="module")
def gn(gpu):
    import gn_bwd
    gn_bwd.lib()
    return gn_bwd


def reference(q, k, v, do, causal, keep):
    """One head in fp64: O, LSE, dQ, dK, dV; a row that sees no key gets zeros and -inf."""
    S, D = q.shape
    sc = (q @ k.t()) * D ** -0.5
    if causal:
        sc.masked_fill_(torch.ones(S, S, device=q.device, dtype=torch.bool).triu(1), -math.inf)
    if keep is not None:
        sc.masked_fill_(~keep[None, :], -math.inf)
    lse = torch.logsumexp(sc, -1)
    p = torch.exp(sc - torch.where(lse == -math.inf, torch.zeros_like(lse), lse)[:, None])
    o = p @ v
    ds = p * (do @ v.t() - (do * o).sum(-1, keepdim=True)) * D ** -0.5
    return o, lse, ds @ k, ds.t() @ q, p.t() @ do


def check(gn, B, H, S, D, causal, mask, grow=0.0, seed=0):
    g = torch.Generator(device="cuda:0")
    g.manual_seed(seed + S + D)
    Q, K, V, dO = (torch.randn(B, H, S, D, device="cuda:0", generator=g) for _ in range(4))
    if grow:  # scores that grow along the keys: the running maximum keeps moving
        K = K + grow * torch.linspace(0, 1, S, device="cuda:0")[:, None] * Q.mean((2,), keepdim=True).sign()
        Q = Q + Q.mean((2,), keepdim=True).sign()
    Q, K, V, dO = (t.bfloat16().contiguous() for t in (Q, K, V, dO))
    O, lse = gn.attn_fwd(Q, K, V, causal=causal, rope="none", mask=mask)
    got = gn.attn_bwd(Q, K, V, O, dO, lse, causal=causal, rope="none", mask=mask)
    refs = [reference(*(t[b, h].double() for t in (Q, K, V, dO)), causal,
                      None if mask is None else mask[b] > 0.5) for b in range(B) for h in range(H)]
    for name, out, j in (("O", O, 0), ("dQ", got[0], 2), ("dK", got[1], 3), ("dV", got[2], 4)):
        ref = torch.stack([r[j] for r in refs]).view(B, H, S, D)
        # one visible key: dQ and dK cancel to 0 and keep the rounding of O in D_i,
        # 2^-9 |dO . O| |K| D^-0.5 < 1e-2 for these unit-variance inputs
        e = float((out.double() - ref).abs().max() / ref.abs().max().clamp(min=1.0))
        assert e < TOL, (name, e)
    ref = torch.stack([r[1] for r in refs]).view(B, H, S)
    dead = ref == -math.inf
    assert bool((lse[dead] == -math.inf).all())
    assert float((lse.double() - ref)[~dead].abs().max()) < 2e-2


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("S", [192, 330, 1000])
def test_masks_with_empty_tiles(gn, D, causal, S):
    keep = torch.ones(5, S)
    keep[1, 64:128] = 0            # a tile in the middle
    keep[2, :70] = 0               # the first tile and a few keys (causal rows that see nothing)
    keep[3] = 0                    # every key
    keep[4, S // 3:] = 0           # a padded end
    keep[4, 3] = 0
    check(gn, 5, 2, S, D, causal, keep.cuda().contiguous())


@pytest.mark.parametrize("causal", [False, True])
def test_more_than_one_window_of_tiles(gn, causal):
    S = 4300
    keep = torch.ones(2, S)
    keep[0, 64 * 60:64 * 66] = 0   # across the 64-tile window
    keep[0, 64 * 66 + 5] = 0
    keep[1, :64 * 64] = 0          # the whole first window
    check(gn, 2, 1, S, 64, causal, keep.cuda().contiguous())


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("S", [1, 63, 65, 127, 129, 961])
def test_ragged_ends_and_growing_maxima(gn, D, S):
    check(gn, 1, 2, S, D, True, None)
    check(gn, 1, 2, S, D, False, None, grow=3.0)
