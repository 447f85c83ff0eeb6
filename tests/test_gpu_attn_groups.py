"""GPU tests of the generic attention path's block shapes: one and two wave groups per block (chosen
by the number of blocks, the sequence length and the head dim), on both sides of each line, with
more blocks than the small cases reach, ragged ends, key masks, and sequences so short that the
second group has no tile.

Sampled heads against 64 bits.  Tolerances as the generic path's other tests (normwise relative):
fp32 1e-4 (two-piece split), bf16 2e-2."""
import math

import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

TOL = {"f32": 1e-4, "bf16": 2e-2}


@pytest.fixture(scope="module")
def gn(gpu):
    import gn_bwd
    gn_bwd.lib()
    return gn_bwd


def rel(a, b):
    return float((a.double() - b).norm() / b.norm().clamp(min=1e-30))


@pytest.mark.parametrize("dt,B,H,S,D,causal,masked", [
    # one group: more than two blocks per CU, two rows of blocks per head, the last one ragged
    ("f32", 5, 60, 130, 32, True, False), ("f32", 5, 60, 130, 64, True, True),
    ("f32", 5, 60, 130, 96, False, False), ("f32", 5, 60, 130, 128, True, True),
    ("bf16", 5, 60, 130, 32, False, True), ("bf16", 5, 60, 130, 96, True, False),
    # and more than that with a long chain
    ("f32", 8, 17, 515, 64, True, False), ("bf16", 8, 17, 515, 96, True, True),
    # 256 and 258 blocks that are not causal, 512 and 514 that are
    ("f32", 2, 64, 256, 64, False, False), ("f32", 3, 43, 256, 64, False, True),
    ("bf16", 2, 64, 256, 96, False, True), ("bf16", 3, 43, 256, 96, False, False),
    ("f32", 8, 32, 256, 96, True, False), ("f32", 1, 257, 256, 96, True, True),
    ("f32", 8, 32, 130, 32, False, False), ("bf16", 8, 32, 256, 32, False, False),
    # two groups: an odd number of tiles, one tile, one tile and a row
    ("f32", 1, 3, 777, 64, True, True), ("f32", 1, 3, 545, 128, False, True),
    ("f32", 1, 3, 300, 128, True, False), ("bf16", 1, 3, 777, 32, True, True),
    ("f32", 2, 2, 31, 64, True, False), ("f32", 2, 2, 33, 96, False, True),
    ("bf16", 2, 2, 31, 96, False, False), ("bf16", 2, 2, 65, 32, True, True),
    ("f32", 1, 2, 65, 128, True, False), ("f32", 1, 1, 1, 64, True, False),
])
def test_groups(gn, dt, B, H, S, D, causal, masked):
    g = torch.Generator(device="cuda:0")
    g.manual_seed(S * D + B)
    ty = torch.float32 if dt == "f32" else torch.bfloat16
    Q, K, V = (torch.randn(B, H, S, D, device="cuda:0", generator=g).to(ty) for _ in range(3))
    dO = (torch.randn(B, H, S, D, device="cuda:0", generator=g) * 0.01).to(ty)
    keep = None
    if masked:  # every batch row keeps its first key, the last one only a few
        keep = torch.ones(B, S, device="cuda:0")
        for b in range(B):
            keep[b, max(1, S - (b + 1) * S // (B + 1)):] = 0.0
    O, lse = gn.attn_fwd(Q, K, V, causal=causal, rope="none", mask=keep)
    grads = gn.attn_bwd(Q, K, V, O, dO, lse, causal=causal, rope="none", mask=keep)
    for h in sorted({0, H // 2, H - 1}):
        for b in sorted({0, B - 1}):
            q, k, v, do = (t[b, h].double() for t in (Q, K, V, dO))
            sc = (q @ k.t().contiguous()) * D ** -0.5
            if causal:
                sc.masked_fill_(torch.ones(S, S, device=sc.device, dtype=torch.bool).triu(1), -math.inf)
            if masked:
                sc.masked_fill_(keep[b] < 0.5, -math.inf)
            p = torch.softmax(sc, -1)
            o = p @ v
            assert rel(O[b, h], o) < TOL[dt]
            assert float((lse[b, h].double() - torch.logsumexp(sc, -1)).abs().max()) < (1e-4 if dt == "f32" else 2e-2)
            ds = p * (do @ v.t().contiguous() - (do * o).sum(-1, keepdim=True)) * D ** -0.5
            # dS = P (dP - D_i) cancels where a row sees one key (S = 1: to zero), and keeps the roundings
            # of both terms: there the size of what cancels is the measure
            both = p * ((do @ v.t().contiguous()).abs() + (do * o).sum(-1, keepdim=True).abs()) * D ** -0.5
            for got, ref, size in zip(grads, (ds @ k, ds.t().contiguous() @ q, p.t().contiguous() @ do),
                                      (both @ k.abs(), both.t().contiguous() @ q.abs(), 0 * q)):
                scale = ref.norm() if S > 1 else torch.maximum(ref.norm(), size.norm())
                assert float((got[b, h].double() - ref).norm() / scale) < TOL[dt]
