"""The measured workloads of this framework: what a program that trains with it calls, over
the range of sizes it calls it with.

Each case is one pass through the public entry points (gn_bwd's functions, grilly_core's tape
through grilly_bridge, decoder_tape.Decoder).  The inputs are seeded and synthetic, with the
distributions the repository's benchmark uses: activations N(0, 1), weights N(0, 0.02),
upstream gradients N(0, 0.01).  Token counts are what a batch happens to hold, so they are
ragged as often as not; feature sizes are the model's.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "grilly-next_amd"))

DEV = "cuda:0"
BF = torch.bfloat16


def listed():
    return [
        # A small fp32 classifier's whole training step through the tape: a handful of launches
        # over tensors of a few kilobytes, so latency and host work are all of it.
        dict(name="mlp_step", kind="mlp", batch=64, din=784, hidden=256, classes=10),
        # An FFN block's forward on the tokens of one short sequence: the weights are read for a
        # few rows.
        dict(name="ffn_fwd_few", kind="ffn_fwd", tokens=37, d=2048, hidden=5632, glu="swiglu_up", bias=False),
        # The same block over a full batch: large products with whole tiles.
        dict(name="ffn_fwd", kind="ffn_fwd", tokens=4096, d=2048, hidden=5632, glu="swiglu_up", bias=False),
        # Its backward, the repository's headline workload.
        dict(name="ffn_bwd", kind="ffn_bwd", tokens=4096, d=2048, hidden=5632, glu="swiglu_up", bias=False),
        # The decoder's FFN (GEGLU, biases) over the tokens left after padding is dropped: a
        # count that no tile divides.
        dict(name="ffn_bwd_ragged", kind="ffn_bwd", tokens=1003, d=768, hidden=3072, glu="geglu_up", bias=True),
        # Causal attention with rotary positions at a training sequence length, forward and
        # backward.
        dict(name="attn", kind="attn", batch=4, heads=16, seq=2048, dim=128, rope="interleaved", causal=True),
        # The decoder's attention over a fused QKV projection with padded sequences (key mask), at a
        # length between the tile sizes.
        dict(name="attn_qkv", kind="attn_qkv", batch=8, heads=12, seq=1000, dim=64, causal=True),
        # fp32 attention (the precision the reference computes in) at an odd length.
        dict(name="attn_f32", kind="attn_f32", batch=2, heads=8, seq=777, dim=64, rope="half", causal=True),
        # The hypervector model's training kernels: unpack-project both ways over packed +-1 inputs
        # and the surrogate loss over K predictions, fp32.
        dict(name="vsa", kind="vsa", rows=8192, out=768, dim=10240, branches=4),
        # The hypernetwork's fp32 output layer at a training batch, forward and backward: a 1 GB
        # weight matrix.
        dict(name="linear_f32", kind="linear_f32", rows=64, din=1536, dout=163840),
        # The end of a language model: final norm, tied head, cross-entropy gradient, their
        # backward and the embedding's, for the tokens of a ragged batch.
        dict(name="lm_head", kind="lm_head", tokens=2001, d=768, vocab=32000),
        # A whole training step of a small decoder: forward, tape backward, AdamW.
        dict(name="decoder_step", kind="decoder", layers=4, batch=8, seq=1024, d=768, heads=12, ff=3072, vocab=32000),
    ]


# ---- ranges --------------------------------------------------------------------------------
def _log(rng, lo, hi):
    """A whole number between lo and hi, spread over the logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["mlp", "ffn_fwd", "ffn_fwd", "ffn_bwd", "ffn_bwd", "attn", "attn_qkv",
                       "attn_f32", "vsa", "linear_f32", "lm_head", "decoder"])
    if kind == "mlp":
        return dict(kind=kind, batch=_log(rng, 8, 2048), din=_log(rng, 64, 1024),
                    hidden=_log(rng, 32, 1024), classes=_log(rng, 2, 128))
    if kind in ("ffn_fwd", "ffn_bwd"):
        # widths are multiples of 64, hidden sizes (often 8/3 of the width) multiples of 8
        d = 64 * rng.randint(4, 32)
        return dict(kind=kind, tokens=_log(rng, 1, 4096), d=d,
                    hidden=8 * rng.randint(2 * d // 8, 11 * d // 32),
                    glu=rng.choice(["swiglu_up", "swiglu_gate", "geglu_up", "geglu_gate", "reglu_up"]),
                    bias=rng.random() < 0.5)
    if kind == "attn":
        return dict(kind=kind, batch=rng.randint(1, 4), heads=rng.randint(2, 16),
                    seq=_log(rng, 64, 2048), dim=rng.choice([64, 64, 96, 128, 128]),
                    rope=rng.choice(["none", "interleaved", "half"]), causal=rng.random() < 0.75)
    if kind == "attn_qkv":
        return dict(kind=kind, batch=rng.randint(1, 8), heads=rng.randint(2, 16),
                    seq=_log(rng, 64, 1400), dim=rng.choice([64, 64, 128]),
                    causal=rng.random() < 0.75)
    if kind == "attn_f32":
        return dict(kind=kind, batch=rng.randint(1, 4), heads=rng.randint(2, 12),
                    seq=_log(rng, 32, 1024), dim=rng.choice([32, 64, 64, 96, 128]),
                    rope=rng.choice(["none", "interleaved", "half"]), causal=rng.random() < 0.75)
    if kind == "vsa":
        return dict(kind=kind, rows=_log(rng, 4, 8192), out=rng.choice([256, 384, 512, 768]),
                    dim=128 * rng.randint(8, 80), branches=rng.randint(2, 4))
    if kind == "linear_f32":
        return dict(kind=kind, rows=_log(rng, 2, 512), din=_log(rng, 64, 1536),
                    dout=_log(rng, 64, 32000))
    if kind == "lm_head":
        return dict(kind=kind, tokens=_log(rng, 16, 2048), d=64 * rng.randint(4, 16),
                    vocab=_log(rng, 1000, 32000))
    heads = rng.randint(4, 12)
    return dict(kind=kind, layers=rng.randint(1, 3), batch=rng.randint(1, 8),
                seq=_log(rng, 64, 1024), d=64 * heads, heads=heads, ff=256 * heads,
                vocab=_log(rng, 1000, 32000))


# ---- inputs --------------------------------------------------------------------------------
def _randn(g, *shape, std=1.0, dtype=torch.float32):
    return (torch.randn(*shape, device=DEV, generator=g) * std).to(dtype).contiguous()


def _glu_fwd(kind, gate, up):
    """glu(gate, up) in plain torch."""
    F = torch.nn.functional
    if kind == "swiglu_up":
        return gate * F.silu(up)
    if kind == "swiglu_gate":
        return F.silu(gate) * up
    if kind == "geglu_up":
        return gate * F.gelu(up, approximate="tanh")
    if kind == "geglu_gate":
        return F.gelu(gate, approximate="tanh") * up
    return gate * F.relu(up)


def prepare(case, seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    kind = case["kind"]
    if kind == "mlp":
        return _prepare_mlp(case, g)
    if kind in ("ffn_fwd", "ffn_bwd"):
        return _prepare_ffn(case, g)
    if kind in ("attn", "attn_qkv", "attn_f32"):
        return _prepare_attn(case, g)
    if kind == "vsa":
        return _prepare_vsa(case, g, seed)
    if kind == "linear_f32":
        R, I, O = case["rows"], case["din"], case["dout"]
        return dict(case=case, X=_randn(g, R, I), W=_randn(g, O, I, std=0.02), b=_randn(g, O, std=0.02),
                    dY=_randn(g, R, O, std=0.01))
    if kind == "lm_head":
        T, d, V = case["tokens"], case["d"], case["vocab"]
        return dict(case=case, x=_randn(g, T, d), gamma=1 + _randn(g, d, std=0.1, dtype=BF),
                    beta=_randn(g, d, std=0.1, dtype=BF), E=_randn(g, V, d, std=0.02, dtype=BF),
                    ids=torch.randint(0, V, (T,), device=DEV, generator=g).to(torch.int32),
                    targets=torch.randint(0, V, (T,), device=DEV, generator=g).to(torch.int32))
    return _prepare_decoder(case, seed)


def _prepare_mlp(case, g):
    import grilly_bridge as gb
    import grilly_core
    B, I, H, C = case["batch"], case["din"], case["hidden"], case["classes"]

    def xavier(o, i):
        lim = math.sqrt(6.0 / (o + i))
        return ((torch.rand(o, i, device=DEV, generator=g) * 2 - 1) * lim).contiguous()

    s = dict(case=case, X=_randn(g, B, I), W1=xavier(H, I), b1=torch.zeros(H, device=DEV),
             W2=xavier(C, H), b2=torch.zeros(C, device=DEV),
             y=torch.randint(0, C, (B,), device=DEV, generator=g).to(torch.int32),
             loss=torch.zeros(1, device=DEV))
    s["device"] = grilly_core.Device(0)
    gb.attach_torch_stream(s["device"])
    s["tape"] = gb.create_tape_context(s["device"], 1 << 20)
    s["opt"] = gb.AdamW([s["W1"], s["b1"], s["W2"], s["b2"]], lr=1e-3)
    return s


def _prepare_ffn(case, g):
    T, d, H = case["tokens"], case["d"], case["hidden"]
    s = dict(case=case, x=_randn(g, T, d, dtype=BF), w=1 + _randn(g, d, std=0.1, dtype=BF),
             Wg=_randn(g, H, d, std=0.02, dtype=BF), Wu=_randn(g, H, d, std=0.02, dtype=BF),
             Wd=_randn(g, d, H, std=0.02, dtype=BF), bg=None, bu=None, bd=None)
    if case["bias"]:
        s.update(bg=_randn(g, H, std=0.02, dtype=BF), bu=_randn(g, H, std=0.02, dtype=BF),
                 bd=_randn(g, d, std=0.02, dtype=BF))
    if case["kind"] == "ffn_bwd":
        # the tensors a forward has saved
        xf = s["x"].float()
        s["rstd"] = torch.rsqrt((xf * xf).mean(-1) + 1e-6).contiguous()
        s["n"] = (xf * s["rstd"][:, None] * s["w"].float()).to(BF).contiguous()

        def lin(x, W, b):
            y = x.float() @ W.float().t()
            return (y if b is None else y + b.float()).to(BF).contiguous()

        s["gate"], s["up"] = lin(s["n"], s["Wg"], s["bg"]), lin(s["n"], s["Wu"], s["bu"])
        s["act"] = _glu_fwd(case["glu"], s["gate"].float(), s["up"].float()).to(BF).contiguous()
        s["dY"] = _randn(g, T, d, std=0.01, dtype=BF)
    return s


def _prepare_attn(case, g):
    B, H, S, D = case["batch"], case["heads"], case["seq"], case["dim"]
    dt = torch.float32 if case["kind"] == "attn_f32" else BF
    s = dict(case=case)
    if case["kind"] == "attn_qkv":
        s["qkv"] = _randn(g, B, S, 3 * H * D, dtype=dt)
        s["dO"] = _randn(g, B, S, H * D, std=0.01, dtype=dt)
        # each sequence is padded at its end: between half and all of its keys are kept
        n = torch.randint((S + 1) // 2, S + 1, (B, 1), device=DEV, generator=g)
        s["mask"] = (torch.arange(S, device=DEV)[None, :] < n).float().contiguous()
    else:
        for k in ("Q", "K", "V"):
            s[k] = _randn(g, B, H, S, D, dtype=dt)
        s["dO"] = _randn(g, B, H, S, D, std=0.01, dtype=dt)
    import gn_bwd as gn
    s["ws"] = gn.workspace(gn.attn_workspace_bytes(B, H, S, D, dt), DEV)
    return s


def _prepare_vsa(case, g, seed):
    R, O, D, K = case["rows"], case["out"], case["dim"], case["branches"]

    def bits():
        return torch.randint(-2**31, 2**31, (R, D // 32), device=DEV, generator=g).to(torch.int32)

    return dict(case=case, seed=int(seed), bits=bits(), target=bits(), W=_randn(g, O, D, std=0.02),
                b=_randn(g, O, std=0.02), dY=_randn(g, R, O), preds=_randn(g, R, K, D))


def _prepare_decoder(case, seed):
    import decoder_tape
    import grilly_bridge as gb
    import grilly_core
    m = decoder_tape.Decoder(case["layers"], case["d"], case["heads"], case["ff"], case["vocab"],
                             case["batch"], case["seq"], int(seed), DEV)
    dev = grilly_core.Device(0)
    gb.attach_torch_stream(dev)
    names = ("ln1_g", "ln1_b", "Wqkv", "bqkv", "Wo", "bo", "ln2_g", "ln2_b", "Wg", "bg", "Wu", "bu", "Wd", "bd")
    weights = [m.E, m.lnf_g, m.lnf_b] + [p[k] for p in m.layers for k in names]
    return dict(case=case, model=m, device=dev, tape=gb.create_tape_context(dev), opt=gb.AdamW(weights, lr=1e-5),
                names=names)


# ---- one pass ------------------------------------------------------------------------------
def run(s):
    return {"mlp": _run_mlp, "ffn_fwd": _run_ffn_fwd, "ffn_bwd": _run_ffn_bwd, "attn": _run_attn,
            "attn_f32": _run_attn, "attn_qkv": _run_attn_qkv, "vsa": _run_vsa,
            "linear_f32": _run_linear, "lm_head": _run_head, "decoder": _run_decoder}[s["case"]["kind"]](s)


def _run_mlp(s):
    """Forward, tape backward and AdamW; the first moments hold the step's gradients."""
    import gn_bwd as gn
    import grilly_bridge as gb
    import grilly_core
    Z = gn.linear_fwd(s["X"], s["W1"], s["b1"])
    H = gn.act_fwd("relu", Z)
    L = gn.linear_fwd(H, s["W2"], s["b2"])
    op, tape = grilly_core.OpType, s["tape"]
    tape.begin()
    n = tape.record_op(op.Linear, [gb.tref(s["X"])], [gb.tref(Z)])
    tape.save_for_backward(n, [s["W1"].data_ptr(), s["b1"].data_ptr()])
    tape.record_op(op.ReLU, [gb.tref(Z, True)], [gb.tref(H)])
    n = tape.record_op(op.Linear, [gb.tref(H, True)], [gb.tref(L)])
    tape.save_for_backward(n, [s["W2"].data_ptr(), s["b2"].data_ptr()])
    n = tape.record_op(op.CrossEntropy, [gb.tref(L, True), gb.tref(s["y"])], [gb.tref(s["loss"])],
                       gb.cross_entropy_params(1.0 / s["case"]["batch"]))
    tape.backward(n, 0)
    s["opt"].step(tape)
    tape.end()
    return dict(logits=L, weights=s["opt"].masters, moments=s["opt"].m)


def _run_ffn_fwd(s):
    import gn_bwd as gn
    n, rstd = gn.rmsnorm_fwd(s["x"], s["w"], eps=1e-6)
    gate, up, act = gn.glu_linear_fwd(s["case"]["glu"], n, s["Wg"], s["Wu"], s["bg"], s["bu"])
    y = gn.linear_fwd(act, s["Wd"], s["bd"])
    return dict(n=n, rstd=rstd, gate=gate, up=up, act=act, y=y)


def _run_ffn_bwd(s):
    import gn_bwd as gn
    bias = s["case"]["bias"]
    gu, dWd, dbd = gn.ffn_down_glu_bwd(s["case"]["glu"], s["dY"], s["act"], s["Wd"], s["gate"], s["up"],
                                       need_db=bias, ws=None)
    dN, dWg, dWu, dbg, dbu = gn.glu_proj_bwd(gu, s["n"], s["Wg"], s["Wu"], need_db=bias, ws=None)
    dx, dw = gn.rmsnorm_bwd(dN, s["x"], s["w"], s["rstd"])
    return dict(dx=dx, dw=dw, dWg=dWg, dWu=dWu, dWd=dWd, dbg=dbg, dbu=dbu, dbd=dbd)


def _run_attn(s):
    import gn_bwd as gn
    kw = dict(causal=s["case"]["causal"], rope=s["case"]["rope"], ws=s["ws"])
    O, lse = gn.attn_fwd(s["Q"], s["K"], s["V"], **kw)
    dQ, dK, dV = gn.attn_bwd(s["Q"], s["K"], s["V"], O, s["dO"], lse, **kw)
    return dict(O=O, lse=lse, dQ=dQ, dK=dK, dV=dV)


def _run_attn_qkv(s):
    """The decoder's attention node: heads split for the forward, the backward on the fused rows."""
    import gn_bwd as gn
    c = s["case"]
    B, H, S, D = c["batch"], c["heads"], c["seq"], c["dim"]
    q, k, v = (t.contiguous() for t in s["qkv"].view(B, S, 3, H, D).permute(2, 0, 3, 1, 4))
    O, lse = gn.attn_fwd(q, k, v, causal=c["causal"], rope="none", ws=s["ws"], mask=s["mask"])
    o = O.permute(0, 2, 1, 3).reshape(B, S, H * D).contiguous()
    dqkv = gn.attn_bwd_qkv(s["qkv"], o, s["dO"], lse, H, causal=c["causal"], rope="none", ws=s["ws"],
                           mask=s["mask"])
    return dict(o=o, lse=lse, dqkv=dqkv)


def _run_vsa(s):
    import gn_bwd as gn
    Y = gn.vsa_unpack_project_fwd(s["bits"], s["W"], s["b"])
    dots, results, weights, loss = gn.vsa_surrogate_fwd(s["preds"], s["target"], seed=s["seed"], counter=1)
    dP = gn.vsa_surrogate_bwd(s["preds"], s["target"], results, weights)
    dW, db = gn.vsa_unpack_project_bwd(s["dY"], s["bits"], s["case"]["dim"])
    # a result row is {winner, runner-up, their dot products as fp32 bits}
    return dict(Y=Y, dots=dots, picked=results[:, :2], picked_dots=results.view(torch.float32)[:, 2:],
                weights=weights, loss=loss, dP=dP, dW=dW, db=db)


def _run_linear(s):
    import gn_bwd as gn
    Y = gn.linear_fwd(s["X"], s["W"], s["b"])
    dX, dW, db = gn.linear_bwd(s["dY"], s["X"], s["W"])
    return dict(Y=Y, dX=dX, dW=dW, db=db)


def _run_head(s):
    import gn_bwd as gn
    T, V = s["case"]["tokens"], s["case"]["vocab"]
    n, mean, rstd = gn.layernorm_fwd(s["x"], s["gamma"], s["beta"], out_dtype=BF)
    logits = gn.linear_fwd(n, s["E"])
    dL = gn.xent_bwd(logits, s["targets"], scale=1.0 / T)
    dn, dE, _ = gn.linear_bwd(dL, n, s["E"], need_db=False)
    dx, dg, db = gn.layernorm_bwd(dn, s["x"], s["gamma"], mean, rstd)
    gn.embedding_bwd(dx, s["ids"], V, dE=dE, accumulate=True)
    return dict(n=n, logits=logits, dL=dL, dx=dx, dE=dE, dgamma=dg, dbeta=db)


def _run_decoder(s):
    """Forward, tape backward and AdamW; the first moments hold the step's gradients."""
    m, tape = s["model"], s["tape"]
    m.forward()
    tape.set_glu_epilogue(m.glu_epilogue)
    tape.begin()
    loss = m.record(tape)
    tape.backward(loss, 0)
    s["opt"].step(tape)
    tape.end()
    return dict(logits=m.logits, moments=s["opt"].m)


# ---- what a pass cannot do without ---------------------------------------------------------
def work(case):
    k = case["kind"]
    if k == "mlp":
        B, I, H, C = case["batch"], case["din"], case["hidden"], case["classes"]
        W = I * H + H + H * C + C
        # inputs and activations once; weights and both moments read and written
        return dict(bytes=4 * (B * I + B * C + 6 * W), flops=2 * B * (2 * I * H + 3 * H * C))
    if k == "ffn_fwd":
        T, d, H = case["tokens"], case["d"], case["hidden"]
        return dict(bytes=2 * (3 * T * d + 3 * T * H + 3 * d * H) + 4 * T, flops=6 * T * d * H)
    if k == "ffn_bwd":
        T, d, H = case["tokens"], case["d"], case["hidden"]
        # reads dY, act, gate, up, n, x and the weights; writes dx and the fp32 weight gradients
        return dict(bytes=2 * (4 * T * d + 3 * T * H + 3 * d * H) + 4 * 3 * d * H, flops=12 * T * d * H)
    if k in ("attn", "attn_qkv", "attn_f32"):
        B, H, S, D = case["batch"], case["heads"], case["seq"], case["dim"]
        e = 4 if k == "attn_f32" else 2
        half = 0.5 if case["causal"] else 1.0
        # Q, K, V, dO read; O, dQ, dK, dV and the row statistics written; 2 products forward, 5 back
        return dict(bytes=8 * e * B * H * S * D + 4 * B * H * S, flops=7 * 2.0 * S * S * D * half * B * H)
    if k == "vsa":
        R, O, D, K = case["rows"], case["out"], case["dim"], case["branches"]
        return dict(bytes=4 * (2 * R * K * D + 2 * R * O + 2 * O * D) + 2 * R * D // 8,
                    flops=4.0 * R * O * D + 6.0 * R * K * D)
    if k == "linear_f32":
        R, I, O = case["rows"], case["din"], case["dout"]
        return dict(bytes=4 * (2 * O * I + 2 * R * I + 2 * R * O + 2 * O), flops=6.0 * R * I * O)
    if k == "lm_head":
        T, d, V = case["tokens"], case["d"], case["vocab"]
        # logits and their gradient are outputs of the pass
        return dict(bytes=2 * 2 * T * V + 2 * V * d + 4 * V * d + 2 * T * d + 2 * 4 * T * d, flops=6.0 * T * d * V)
    L, T, S, d, ff, V = (case["layers"], case["batch"] * case["seq"], case["seq"], case["d"], case["ff"],
                         case["vocab"])
    per = 4 * d * d + 3 * d * ff
    W = L * per + V * d
    # weights: bf16 read and written, fp32 master and both moments read and written; logits out
    return dict(bytes=28 * W + 2 * T * V,
                flops=6.0 * T * W + L * 7 * 2.0 * S * S * d * 0.5 * case["batch"])


def tolerance(case):
    """Largest relative differences between correct implementations of the same precision: about
    four times the largest error against 64 bits measured over the listed and some drawn cases."""
    k = case["kind"]
    if k in ("ffn_fwd", "attn"):
        return {"rel": 1.6e-2}  # bf16 results and probabilities: 4.3e-3, 3.7e-3
    if k in ("ffn_bwd", "attn_qkv", "lm_head"):
        return {"rel": 1.2e-2}  # bf16 gradients between the products: 2.9e-3, 2.4e-3, 2.4e-3
    if k == "decoder":
        return {"rel": 4e-2}  # bf16 activations through every layer, both ways: 1.0e-2
    if k == "attn_f32":
        return {"rel": 4e-5}  # fp32 as two bf16 pieces per operand: 8e-6
    # fp32 sums: 2.6e-6 (a packed sum of 10240 terms); winners of the selection may tie
    return {"rel": 1e-5, "differ": 1e-3}


# ---- 64-bit results ------------------------------------------------------------------------
def exact(case, seed):
    s = prepare(case, seed)
    return {"mlp": _exact_mlp, "ffn_fwd": _exact_ffn_fwd, "ffn_bwd": _exact_ffn_bwd, "attn": _exact_attn,
            "attn_f32": _exact_attn, "attn_qkv": _exact_attn_qkv, "vsa": _exact_vsa,
            "linear_f32": _exact_linear, "lm_head": _exact_head, "decoder": _exact_decoder}[case["kind"]](s)


def _d(t):
    return None if t is None else t.double()


def _lin(x, W, b):
    y = x @ W.t()
    return y if b is None else y + b


def _adamw(W, g, lr):
    """The first AdamW step (betas 0.9 / 0.999, eps 1e-8, weight decay 0.01) and its first moment."""
    return W * (1 - lr * 0.01) - lr * g / (g.abs() + 1e-8), 0.1 * g


def _exact_mlp(s):
    X, W1, b1, W2, b2 = (_d(s[k]) for k in ("X", "W1", "b1", "W2", "b2"))
    Z = X @ W1.t() + b1
    H = Z.clamp(min=0)
    L = H @ W2.t() + b2
    dL = torch.softmax(L, -1)
    dL[torch.arange(len(dL), device=DEV), s["y"].long()] -= 1
    dL = dL / len(dL)
    dZ = (dL @ W2) * (Z > 0)
    new = [_adamw(W, g, 1e-3) for W, g in ((W1, dZ.t() @ X), (b1, dZ.sum(0)), (W2, dL.t() @ H), (b2, dL.sum(0)))]
    return dict(logits=L, weights=[w for w, _ in new], moments=[m for _, m in new])


def _exact_ffn_fwd(s):
    x = _d(s["x"])
    rstd = torch.rsqrt((x * x).mean(-1) + 1e-6)
    n = x * rstd[:, None] * _d(s["w"])
    gate, up = _lin(n, _d(s["Wg"]), _d(s["bg"])), _lin(n, _d(s["Wu"]), _d(s["bu"]))
    act = _glu_fwd(s["case"]["glu"], gate, up)
    return dict(n=n, rstd=rstd, gate=gate, up=up, act=act, y=_lin(act, _d(s["Wd"]), _d(s["bd"])))


def _exact_ffn_bwd(s):
    dY, bias = _d(s["dY"]), s["case"]["bias"]
    gate, up = _d(s["gate"]).requires_grad_(), _d(s["up"]).requires_grad_()
    dG, dU = torch.autograd.grad(_glu_fwd(s["case"]["glu"], gate, up), (gate, up), dY @ _d(s["Wd"]))
    n, x, w, r = _d(s["n"]), _d(s["x"]), _d(s["w"]), _d(s["rstd"])[:, None]
    dN = dG @ _d(s["Wg"]) + dU @ _d(s["Wu"])
    dx = r * w * dN - x * r**3 * (w * dN * x).mean(-1, keepdim=True)
    return dict(dx=dx, dw=(dN * x * r).sum(0), dWg=dG.t() @ n, dWu=dU.t() @ n, dWd=dY.t() @ _d(s["act"]),
                dbg=dG.sum(0) if bias else None, dbu=dU.sum(0) if bias else None,
                dbd=dY.sum(0) if bias else None)


def _rope(x, mode, back=False):
    """Rotary positions 0..S-1 (base 10000) on [S, D]; back: the transposed rotation."""
    if mode == "none":
        return x
    S, D = x.shape
    ang = torch.arange(S, device=DEV, dtype=torch.float64)[:, None] * 10000.0 ** (
        -torch.arange(0, D, 2, device=DEV, dtype=torch.float64) / D)[None, :]
    c, sn = ang.cos(), ang.sin()
    if back:
        sn = -sn
    if mode == "interleaved":
        a, b = x[:, 0::2], x[:, 1::2]
        return torch.stack((a * c - b * sn, a * sn + b * c), -1).reshape(S, D)
    a, b = x[:, :D // 2], x[:, D // 2:]
    return torch.cat((a * c - b * sn, a * sn + b * c), -1)


def _head(q, k, v, do, rope, causal, keep):
    """One head's O, logsumexp, dQ, dK, dV; keep [S]: the keys that are not padding (or None)."""
    S, D = q.shape
    q, k = _rope(q, rope), _rope(k, rope)
    scale = D ** -0.5
    sc = (q @ k.t()) * scale
    if causal:
        sc.masked_fill_(torch.ones(S, S, device=DEV, dtype=torch.bool).triu(1), -math.inf)
    if keep is not None:
        sc.masked_fill_(~keep[None, :], -math.inf)
    lse = torch.logsumexp(sc, -1)
    p = torch.exp(sc - lse[:, None])
    o = p @ v
    dp = do @ v.t()
    ds = p * (dp - (do * o).sum(-1, keepdim=True)) * scale
    return o, lse, _rope(ds @ k, rope, True), _rope(ds.t() @ q, rope, True), p.t() @ do


def _exact_attn(s):
    c = s["case"]
    B, H, S, D = c["batch"], c["heads"], c["seq"], c["dim"]
    flat = [s[k].reshape(B * H, S, D) for k in ("Q", "K", "V", "dO")]
    got = [_head(*(t[i].double() for t in flat), c["rope"], c["causal"], None) for i in range(B * H)]
    O, lse, dQ, dK, dV = (torch.stack([h[j] for h in got]) for j in range(5))
    sh = (B, H, S, D)
    return dict(O=O.view(sh), lse=lse.view(B, H, S), dQ=dQ.view(sh), dK=dK.view(sh), dV=dV.view(sh))


def _exact_attn_qkv(s):
    c = s["case"]
    B, H, S, D = c["batch"], c["heads"], c["seq"], c["dim"]
    qkv, dO = s["qkv"].view(B, S, 3, H, D), s["dO"].view(B, S, H, D)
    o = torch.empty(B, S, H, D, device=DEV, dtype=torch.float64)
    lse = torch.empty(B, H, S, device=DEV, dtype=torch.float64)
    dqkv = torch.empty(B, S, 3, H, D, device=DEV, dtype=torch.float64)
    for b in range(B):
        keep = s["mask"][b] > 0.5
        for h in range(H):
            q, k, v = (qkv[b, :, i, h].double() for i in range(3))
            o[b, :, h], lse[b, h], dqkv[b, :, 0, h], dqkv[b, :, 1, h], dqkv[b, :, 2, h] = _head(
                q, k, v, dO[b, :, h].double(), "none", c["causal"], keep)
    return dict(o=o.view(B, S, H * D), lse=lse, dqkv=dqkv.view(B, S, 3 * H * D))


def _unpack(bits):
    """[R, words] packed -> [R, 32 words] of +-1."""
    sh = torch.arange(32, device=DEV, dtype=torch.int32)
    return (((bits[:, :, None] >> sh) & 1).reshape(len(bits), -1) * 2 - 1).double()


def _gumbel(seed, counter, R, K):
    """The documented counter-based noise of the surrogate selection (splitmix64, 23 bits)."""
    with np.errstate(over="ignore"):
        n = np.uint64(counter) * np.uint64(R) + np.arange(R, dtype=np.uint64)[:, None]
        z = np.uint64(seed) + (n * np.uint64(K) + np.arange(K, dtype=np.uint64)[None, :] + np.uint64(1)) * np.uint64(
            0x9E3779B97F4A7C15)
        z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
        z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
        z = z ^ (z >> np.uint64(31))
    u = ((z >> np.uint64(41)).astype(np.float64) + 0.5) / 2.0**23
    return torch.from_numpy(-np.log(-np.log(u))).to(DEV)


def _exact_vsa(s):
    c = s["case"]
    R, D, K = c["rows"], c["dim"], c["branches"]
    gamma, delta, lam = 1.0, 1.0, 0.3
    bits = _unpack(s["bits"])
    Y = bits @ _d(s["W"]).t() + _d(s["b"])
    dW, db = _d(s["dY"]).t() @ bits, _d(s["dY"]).sum(0)
    del bits
    y = _unpack(s["target"])
    P = s["preds"].double()
    dots = torch.stack([(P[:, k] * y).sum(-1) for k in range(K)], 1)
    noisy = dots + _gumbel(s["seed"], 1, R, K)
    order = noisy.argsort(dim=1, descending=True, stable=True)[:, :2]
    picked = dots.gather(1, order)
    weights = torch.softmax(dots, -1)
    rows = torch.arange(R, device=DEV)
    hinge = (gamma - y * P[rows, order[:, 0]]).clamp(min=0).mean(-1)
    margin = delta - (picked[:, 0] - picked[:, 1])
    loss = hinge + lam * margin.clamp(min=0)
    dP = torch.empty_like(P)
    for k in range(K):
        dP[:, k] = torch.where(gamma - y * P[:, k] > 0, -y / D * weights[:, k:k + 1], torch.zeros_like(y))
    dP[rows, order[:, 1]] += y / D * lam * (margin > 0).double()[:, None]
    return dict(Y=Y, dots=dots, picked=order.to(torch.int32), picked_dots=picked, weights=weights, loss=loss,
                dP=dP, dW=dW, db=db)


def _exact_linear(s):
    X, W, dY = _d(s["X"]), _d(s["W"]), _d(s["dY"])
    return dict(Y=_lin(X, W, _d(s["b"])), dX=dY @ W, dW=dY.t() @ X, db=dY.sum(0))


def _ln(x, gamma, beta):
    mean = x.mean(-1, keepdim=True)
    return (x - mean) * torch.rsqrt(((x - mean) ** 2).mean(-1, keepdim=True) + 1e-5) * gamma + beta


def _exact_head(s):
    T = s["case"]["tokens"]
    x, gamma, beta, E = (_d(s[k]).requires_grad_() for k in ("x", "gamma", "beta", "E"))
    n = _ln(x, gamma, beta)
    logits = n @ E.t()
    dL = torch.softmax(logits.detach(), -1)
    dL[torch.arange(T, device=DEV), s["targets"].long()] -= 1
    dL = dL / T
    dx, dg, db, dE = torch.autograd.grad(logits, (x, gamma, beta, E), dL)
    dE = dE.index_add(0, s["ids"].long(), dx)
    return dict(n=n.detach(), logits=logits.detach(), dL=dL, dx=dx, dE=dE, dgamma=dg, dbeta=db)


def _exact_decoder(s):
    m = s["model"]
    B, S, H, d = m.B, m.S, m.H, m.d
    lay = [{k: _d(p[k]).requires_grad_() for k in s["names"]} for p in m.layers]
    E, fg, fb = (_d(t).requires_grad_() for t in (m.E, m.lnf_g, m.lnf_b))
    later = torch.ones(S, S, device=DEV, dtype=torch.bool).triu(1)
    x = E[m.ids.long()]
    for p in lay:
        q, k, v = _lin(_ln(x, p["ln1_g"], p["ln1_b"]), p["Wqkv"], p["bqkv"]).view(B, S, 3, H, d // H).permute(
            2, 0, 3, 1, 4)
        sc = (q.contiguous() @ k.transpose(-1, -2).contiguous()) * (d // H) ** -0.5
        o = torch.softmax(sc.masked_fill(later, -math.inf), -1) @ v.contiguous()
        x = x + _lin(o.permute(0, 2, 1, 3).reshape(B * S, d), p["Wo"], p["bo"])
        n = _ln(x, p["ln2_g"], p["ln2_b"])
        h = _glu_fwd("geglu_up", _lin(n, p["Wg"], p["bg"]), _lin(n, p["Wu"], p["bu"]))
        x = x + _lin(h, p["Wd"], p["bd"])
    logits = _ln(x, fg, fb) @ E.t()
    dL = torch.softmax(logits.detach(), -1)
    dL[torch.arange(B * S, device=DEV), m.tgt.long()] -= 1
    weights = [E, fg, fb] + [p[k] for p in lay for k in s["names"]]
    grads = torch.autograd.grad(logits, weights, dL / (B * S))
    return dict(logits=logits.detach(), moments=[0.1 * g for g in grads])
