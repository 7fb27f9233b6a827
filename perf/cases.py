"""The work a program has this library do, as cases that can be timed and compared.

A case is a dict of plain values.  `listed()` gives the standing ones, `draw(rng)` more of
the same ranges, `prepare` the device buffers a caller holds before the call, `run` one pass
through the public entry points, `work` what that pass cannot do without, `tolerance` how
far two correct implementations may differ and `exact` the same results in 64 bits, in plain
torch.

Kinds of case (the sizes are those of the library's own benchmark and tests, or generic):
  step       one greedy decode step of a hybrid decoder for a batch of sequences, replayed
             as a HIP graph the way a serving loop runs it
  mlp        the SwiGLU MLP over a few decode rows or a chunk of prompt rows
  gemv       one projection (K-quant rows or packed tiles, or a float matrix)
  lm_head    vocabulary readout and margin argmax
  attention  decode attention over quantised history packets
  delta      one token through a gated delta-net layer's own ops
  pack       the load-time repacking of a matrix for the matrix cores
"""
import math
import os
import random
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "ray-tracing-attention_amd"))
from rta import _lib, model, ops  # noqa: E402

FMT = {"f32": _lib.F32, "f16": _lib.F16, "bf16": _lib.BF16, "q4k": _lib.Q4_K, "q6k": _lib.Q6_K}
BLOCK = {"q4k": 144, "q6k": 210}
HD = 128
DEV = "cuda:0"


def listed():
    return [
        # the headline workload: the 9B-shaped step for one sequence (GGUF rows) and for a
        # continuous batch of 32 (packed tiles), contexts of 256 to 8192 tokens
        step_case("step_9b_b1", 1, 32, 4096, 32, 8, 32, 12288, 151936, False, 256, 8192),
        step_case("step_9b_b32", 32, 32, 4096, 32, 8, 32, 12288, 151936, True, 256, 8192),
        # a small decoder serving more sequences than one matrix-core batch tile
        step_case("step_2048_b64", 64, 8, 2048, 16, 4, 16, 6144, 32000, True, 64, 2048),
        # one projection of one token: the smallest call, bound by latency
        dict(name="gemv_q4k_4096_b1", kind="gemv", fmt="q4k", packed=False, rows=4096, cols=4096, batch=1,
             accumulate=False),
        # a ragged residual projection of a few sequences, GGUF rows, added into the stream
        dict(name="gemv_q6k_5003x1280_b3", kind="gemv", fmt="q6k", packed=False, rows=5003, cols=1280, batch=3,
             accumulate=True),
        # the small model's MLP as its file holds it, for a batch of 8 rows
        dict(name="mlp_2048_b8", kind="mlp", fmt_d="q6k", packed=False, hidden=2048, inter=6144, batch=8,
             accumulate=False),
        # the 9B MLP over a chunk of prompt rows (prefill), packed tiles
        dict(name="mlp_4096_b256", kind="mlp", fmt_d="q4k", packed=True, hidden=4096, inter=12288, batch=256,
             accumulate=True),
        # the vocabulary readout of 4 sequences from the exported Q6_K rows
        dict(name="lm_head_2048_b4", kind="lm_head", fmt="q6k", packed=False, vocab=151936, hidden=2048, batch=4),
        # 16 sequences with ragged contexts, grouped heads, Q6_K keys and Q4_K values
        dict(name="attention_gqa_16seq", kind="attention", hq=16, hkv=4, fmt_k="q6k", fmt_v="q4k", nseq=16,
             ctx_lo=512, ctx_hi=32768, capacity=32768, gate=False),
        # one long conversation over the reference's packet layout, with the output gate
        dict(name="attention_long", kind="attention", hq=32, hkv=8, fmt_k="q4k", fmt_v="q6k", nseq=1,
             ctx_lo=100003, ctx_hi=100003, capacity=131072, gate=True),
        # the delta-net ops of a layer for 32 sequences, called one by one
        dict(name="delta_b32", kind="delta", batch=32, heads=32),
        # loading a model: the LM head's rows into packed tiles
        dict(name="pack_q6k_lm_head", kind="pack", fmt="q6k", rows=151936, cols=2048),
    ]


def step_case(name, batch, layers, hidden, q_heads, kv_heads, rec_heads, ff, vocab, packed, ctx_lo, ctx_hi):
    c = dict(kind="step", batch=batch, layers=layers, hidden=hidden, q_heads=q_heads, kv_heads=kv_heads,
             rec_heads=rec_heads, ff=ff, vocab=vocab, packed=packed, ctx_lo=ctx_lo, ctx_hi=ctx_hi)
    return dict(c, name=name) if name else c


# ------------------------------------------------------------------ drawn cases ----
def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _blocks(rng, lo, hi):
    """A multiple of 256 between lo and hi, spread over its logarithm."""
    return 256 * _log_int(rng, lo // 256, hi // 256)


def draw(rng):
    kind = rng.choice(["step", "mlp", "mlp", "gemv", "gemv", "gemv", "lm_head", "attention", "attention", "delta",
                       "pack"])
    if kind == "step":
        heads = rng.choice([(8, 2), (16, 4), (16, 8)])
        return step_case(None, _log_int(rng, 1, 64), rng.choice([4, 8]), rng.choice([1024, 1536, 2048]), *heads,
                         rng.choice([8, 16]), _blocks(rng, 1024, 6144), _log_int(rng, 4000, 32000),
                         rng.random() < 0.6, 32, _log_int(rng, 64, 4096))
    if kind == "mlp":
        return dict(kind=kind, fmt_d=rng.choice(["q4k", "q6k"]), packed=rng.random() < 0.5,
                    hidden=_blocks(rng, 512, 4096), inter=_blocks(rng, 1024, 12288), batch=_log_int(rng, 1, 256),
                    accumulate=rng.random() < 0.5)
    if kind == "gemv":
        fmt = rng.choice(["q4k", "q4k", "q4k", "q6k", "q6k", "f32", "f16", "bf16"])
        if fmt in BLOCK:
            return dict(kind=kind, fmt=fmt, packed=rng.random() < 0.5, rows=_log_int(rng, 64, 16448),
                        cols=_blocks(rng, 512, 12288), batch=_log_int(rng, 1, 192), accumulate=rng.random() < 0.5)
        # float matrices are the small ones of a model (decay and write-strength rows)
        return dict(kind=kind, fmt=fmt, packed=False, rows=_log_int(rng, 16, 1024),
                    cols=4 * _log_int(rng, 64, 1024), batch=_log_int(rng, 1, 32), accumulate=rng.random() < 0.5)
    if kind == "lm_head":
        return dict(kind=kind, fmt=rng.choice(["q4k", "q6k"]), packed=rng.random() < 0.5,
                    vocab=_log_int(rng, 4000, 151936), hidden=_blocks(rng, 1024, 4096), batch=_log_int(rng, 1, 48))
    if kind == "attention":
        hq, hkv = rng.choice([(16, 4), (32, 8), (8, 8), (16, 2), (4, 4), (24, 6)])
        fmt_k, fmt_v = rng.choice([("q4k", "q6k"), ("q4k", "q6k"), ("q6k", "q4k"), ("q4k", "q4k")])
        nseq = _log_int(rng, 1, 64)
        hi = _log_int(rng, 64, min(65536, 400000 // nseq))
        return dict(kind=kind, hq=hq, hkv=hkv, fmt_k=fmt_k, fmt_v=fmt_v, nseq=nseq,
                    ctx_lo=max(1, hi // rng.choice([1, 8, 64])), ctx_hi=hi,
                    capacity=hi if rng.random() < 0.7 else max(32, hi - hi // 5), gate=rng.random() < 0.5)
    if kind == "delta":
        return dict(kind=kind, batch=_log_int(rng, 1, 64), heads=rng.choice([8, 16, 24, 32]))
    return dict(kind=kind, fmt=rng.choice(["q4k", "q6k"]), rows=_log_int(rng, 100, 40000), cols=_blocks(rng, 512, 4096))


# ----------------------------------------------------------------------- inputs ----
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) & 0x7fffffffffffffff)
    return g


def _randn(shape, g, scale=1.0):
    return torch.randn(*shape, device=DEV, generator=g) * scale


def _matrix(case, fmt, rows, cols, g):
    """The matrix in its file's format and as the call takes it (packed when asked)."""
    if fmt not in BLOCK:
        w = model.random_float_matrix(FMT[fmt], rows, cols, g, torch.device(DEV))
        return w, w, FMT[fmt]
    w = model.random_kquant(FMT[fmt], rows, cols, g, torch.device(DEV))
    if not case.get("packed"):
        return w, w, FMT[fmt]
    return w, ops.pack(FMT[fmt], w, rows, cols), FMT[fmt] | ops.TILED


def _contexts(case, n):
    """Ragged context lengths, log-uniform, fixed by the case: they are its size."""
    r = random.Random(f"{case['ctx_lo']} {case['ctx_hi']} {n}")
    lo, hi = case["ctx_lo"], case["ctx_hi"]
    return [min(hi, max(lo, int(math.exp(r.uniform(math.log(lo), math.log(hi + 1)))))) for _ in range(n)]


def _packets(n, kvw, fmt_k, fmt_v, g):
    """n history packets with random codes and the block scales quantised activations have."""
    nb = (kvw + 255) // 256
    pk = torch.zeros(n, ops.history_bytes(kvw), dtype=torch.uint8, device=DEV)
    pk.random_(0, 256, generator=g)
    half = lambda: (torch.rand(n, device=DEV, generator=g) * 0.01 + 1e-3).half().view(torch.uint8).view(n, 2)  # noqa: E731
    at = 0
    for fmt in (fmt_k, fmt_v):
        for _ in range(nb):
            if fmt == "q4k":
                pk[:, at:at + 2], pk[:, at + 2:at + 4] = half(), half()
            else:
                pk[:, at + 192:at + 208] = torch.randint(-32, 32, (n, 16), dtype=torch.int8, device=DEV,
                                                         generator=g).view(torch.uint8)
                pk[:, at + 208:at + 210] = half()
            at += BLOCK[fmt]
    pk[:, at:] = 0
    return pk


def _decode_model(case, seed, packed, keep=False):
    q4, q6, tiled = _lib.Q4_K, _lib.Q6_K, _lib.TILED if packed else 0
    s = model.HybridShape(hidden=case["hidden"], layers=case["layers"], full_every=4, q_heads=case["q_heads"],
                          kv_heads=case["kv_heads"], head_dim=HD, rec_heads=case["rec_heads"], ff=case["ff"],
                          vocab=case["vocab"], capacity=case["ctx_hi"] + 256, fmt_embed=q4, fmt_proj=q4 | tiled,
                          fmt_lm=q6 | tiled, fmt_k=q4, fmt_v=q6, rope_rotary=HD, eps=1e-6, margin=1e-4,
                          rope_theta=1e6)
    return model.DecodeModel(s, case["batch"], _contexts(case, case["batch"]), seed=int(seed), dev=DEV,
                             keep_gguf=keep)


def _state_part(m, which):
    """A view of the model's recurrent or conv state or of its history packets."""
    s, v = m.shape, m.views
    nfull = s.layers // s.full_every
    nrec = s.layers - nfull
    if which == "packets":
        at, n = v.packets - m.state.data_ptr(), nfull * v.slots_per_layer * v.packet_bytes
        return m.state[at:at + n].view(nfull, m.batch, s.capacity, v.packet_bytes)
    per, ptr = (v.recurrent_per_layer, v.recurrent) if which == "recurrent" else (v.conv_per_layer, v.conv)
    at = ptr - m.state.data_ptr()
    f = m.state[at:at + 4 * nrec * per].view(torch.float32)
    if which == "recurrent":
        return f.view(nrec, m.batch, s.rec_heads, HD, HD)
    return f.view(nrec, m.batch, 3 * s.rec_heads * HD, 3)


def prepare(case, seed):
    g, kind = _gen(seed), case["kind"]
    if kind == "step":
        m = _decode_model(case, seed, case["packed"])
        # one eager step loads the kernels; then the state is put back and the step captured
        kept = [(t, t.clone()) for t in (_state_part(m, "recurrent"), _state_part(m, "conv"), m.tokens)]
        m.step(logits=True)
        for t, was in kept:
            t.copy_(was)
        _lib.check(m.lib.rta_hybrid_init(m.shape, m.batch, m.state.data_ptr(), m.ctx.data_ptr(), ops._stream()))
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            m.step(logits=True)
        return dict(kind=kind, m=m, graph=graph,
                    out=dict(logits=m.logits, tokens=m.tokens, recurrent=_state_part(m, "recurrent"),
                             conv=_state_part(m, "conv"), packets=_state_part(m, "packets")))
    if kind == "gemv":
        raw, w, fmt = _matrix(case, case["fmt"], case["rows"], case["cols"], g)
        b = case["batch"]
        x, y = _randn((b, case["cols"]), g), _randn((b, case["rows"]), g)
        ws = torch.empty(ops.gemv_workspace_bytes(fmt, case["rows"], case["cols"], b) or 1, dtype=torch.uint8, device=DEV)
        return dict(kind=kind, case=case, raw=raw, w=w, fmt=fmt, x=x, y=y, ws=ws)
    if kind == "mlp":
        h, n, b = case["hidden"], case["inter"], case["batch"]
        gate, up, down = (_matrix(case, f, r, c, g) for f, r, c in (("q4k", n, h), ("q4k", n, h), (case["fmt_d"], h, n)))
        x, y = _randn((b, h), g), _randn((b, h), g)
        act = torch.empty(b, n, device=DEV)
        fmts = (gate[2], up[2], down[2])
        ws = torch.empty(ops.mlp_workspace_bytes(fmts[0], fmts[2], h, n, b) or 1, dtype=torch.uint8, device=DEV)
        return dict(kind=kind, case=case, raw=[t[0] for t in (gate, up, down)], w=[t[1] for t in (gate, up, down)],
                    fmts=fmts, x=x, y=y, act=act, ws=ws)
    if kind == "lm_head":
        raw, w, fmt = _matrix(case, case["fmt"], case["vocab"], case["hidden"], g)
        b = case["batch"]
        h = _randn((b, case["hidden"]), g, 2.0)
        ws = torch.empty(ops.lm_head_workspace_bytes(fmt, case["vocab"], case["hidden"], b), dtype=torch.uint8, device=DEV)
        return dict(kind=kind, case=case, raw=raw, w=w, fmt=fmt, h=h, ws=ws,
                    logits=torch.empty(b, case["vocab"], device=DEV), ids=torch.empty(b, dtype=torch.int32, device=DEV))
    if kind == "attention":
        n, cap = case["nseq"], case["capacity"]
        ctx = _contexts(case, n)
        held = [min(c, cap) for c in ctx]
        # every sequence owns a ring of `capacity` slots; only the slots in use exist here
        base, at = [], 0
        for c, used in zip(ctx, held):
            base.append(at)
            at += cap if c > cap else used
        packets = _packets(at, case["hkv"] * HD, case["fmt_k"], case["fmt_v"], g)
        q = _randn((n, case["hq"], HD), g)
        gate = _randn((n, case["hq"], HD), g) if case["gate"] else None
        need = ops.decode_attention_workspace_bytes(n, case["hq"], case["hkv"], HD, max(held))
        return dict(kind=kind, case=case, q=q, gate=gate, packets=packets, max_ctx=max(held),
                    base=torch.tensor(base, dtype=torch.int64, device=DEV),
                    ctx=torch.tensor(ctx, dtype=torch.int32, device=DEV), out=torch.empty_like(q),
                    ws=torch.empty(need, dtype=torch.uint8, device=DEV))
    if kind == "delta":
        b, h = case["batch"], case["heads"]
        w = h * HD
        proj = _randn((b, 4 * w + 2 * h), g)
        target = 0.9 + 0.099 * torch.rand(h, device=DEV, generator=g)
        dt = 2.0 * torch.rand(h, device=DEV, generator=g) - 1.0
        return dict(kind=kind, case=case, proj=proj, conv=_randn((b, 3 * w, 3), g), taps=_randn((3 * w, 4), g, 0.5),
                    a_log=torch.log(-torch.log(target) / torch.nn.functional.softplus(dt)), dt_bias=dt,
                    state=_randn((b, h, HD, HD), g, 0.1), norm=1.0 + _randn((w,), g, 0.05),
                    qkv=torch.empty(b, 3 * w, device=DEV), decay=torch.empty(b, h, device=DEV),
                    beta=torch.empty(b, h, device=DEV), out=torch.empty(b, w, device=DEV))
    assert kind == "pack"
    return dict(kind=kind, case=case, w=model.random_kquant(FMT[case["fmt"]], case["rows"], case["cols"], g,
                                                            torch.device(DEV)))


# --------------------------------------------------------------------- one pass ----
def run(state):
    kind, c = state["kind"], state.get("case")
    if kind == "step":
        state["graph"].replay()
        return state["out"]
    if kind == "gemv":
        return ops.gemv(state["fmt"], state["w"], c["rows"], c["cols"], state["x"], y=state["y"],
                        accumulate=c["accumulate"], workspace=state["ws"])
    if kind == "mlp":
        return ops.mlp_swiglu(state["fmts"], *state["w"], c["hidden"], c["inter"], state["x"], y=state["y"],
                              accumulate=c["accumulate"], act=state["act"], workspace=state["ws"])
    if kind == "lm_head":
        return ops.lm_head(state["fmt"], state["w"], c["vocab"], c["hidden"], state["h"], workspace=state["ws"],
                           logits=state["logits"], ids=state["ids"])
    if kind == "attention":
        return ops.decode_attention(state["q"], state["packets"], FMT[c["fmt_k"]], FMT[c["fmt_v"]], state["base"],
                                    state["ctx"], c["capacity"], state["max_ctx"], c["hkv"], gate=state["gate"],
                                    workspace=state["ws"], out=state["out"])
    if kind == "delta":
        h = c["heads"]
        w = h * HD
        p = state["proj"]
        ops.short_conv(p[:, :3 * w], state["conv"], state["taps"], h, out=state["qkv"])
        ops.delta_gates(p[:, 4 * w:4 * w + h], p[:, 4 * w + h:], state["a_log"], state["dt_bias"],
                        decay=state["decay"], beta=state["beta"])
        out = ops.delta_rule(state["state"], state["qkv"], state["decay"], state["beta"], h, norm_w=state["norm"],
                             gate=p[:, 3 * w:4 * w], out=state["out"])
        return dict(out=out, conv=state["conv"], state=state["state"])
    return ops.pack(FMT[c["fmt"]], state["w"], c["rows"], c["cols"])


# ------------------------------------------------------------ what a pass needs ----
def _weight_bytes(fmt, rows, cols):
    return rows * (cols // 256) * BLOCK[fmt] if fmt in BLOCK else rows * cols * (4 if fmt == "f32" else 2)


def _step_sizes(c):
    nfull = c["layers"] // 4
    nrec = c["layers"] - nfull
    s = c["rec_heads"] * HD
    rows_full, rows_rec = (c["q_heads"] + 2 * c["kv_heads"]) * HD, 4 * s + 2 * c["rec_heads"]
    weights = (nfull * (rows_full * c["hidden"] + c["hidden"] * c["q_heads"] * HD) +
               nrec * (rows_rec * c["hidden"] + c["hidden"] * s) + 3 * c["layers"] * c["hidden"] * c["ff"])
    return nfull, nrec, s, weights


def work(case):
    kind = case["kind"]
    if kind == "step":
        nfull, nrec, s, weights = _step_sizes(case)
        b, kvw = case["batch"], case["kv_heads"] * HD
        seen = sum(x + 1 for x in _contexts(case, b))
        lm = case["vocab"] * case["hidden"]
        packet = 8 * ((kvw + 255) // 256 * 354 // 8 + 1)
        state = nrec * b * (case["rec_heads"] * HD * HD + 9 * s) * 4 * 2
        return {"bytes": weights // 256 * 144 + lm // 256 * 210 + nfull * seen * packet + state + 4 * b * case["vocab"],
                "flops": 2.0 * b * (weights + lm) + 4.0 * nfull * seen * case["q_heads"] * HD +
                nrec * b * case["rec_heads"] * HD * HD * 7.0}
    if kind == "gemv":
        r, c, b = case["rows"], case["cols"], case["batch"]
        return {"bytes": _weight_bytes(case["fmt"], r, c) + 4 * b * (c + r * (2 if case["accumulate"] else 1)),
                "flops": 2.0 * r * c * b}
    if kind == "mlp":
        h, n, b = case["hidden"], case["inter"], case["batch"]
        return {"bytes": 2 * _weight_bytes("q4k", n, h) + _weight_bytes(case["fmt_d"], h, n) +
                4 * b * (h + n + h * (2 if case["accumulate"] else 1)), "flops": 6.0 * h * n * b}
    if kind == "lm_head":
        v, h, b = case["vocab"], case["hidden"], case["batch"]
        return {"bytes": _weight_bytes(case["fmt"], v, h) + 4 * b * (h + v), "flops": 2.0 * v * h * b}
    if kind == "attention":
        kvw = case["hkv"] * HD
        seen = sum(min(x, case["capacity"]) for x in _contexts(case, case["nseq"]))
        per = (kvw + 255) // 256 * (BLOCK[case["fmt_k"]] + BLOCK[case["fmt_v"]])
        rows = case["nseq"] * case["hq"] * HD
        return {"bytes": seen * per + 4 * rows * (3 if case["gate"] else 2), "flops": 4.0 * seen * case["hq"] * HD}
    if kind == "delta":
        b, w = case["batch"], case["heads"] * HD
        return {"bytes": 4 * b * (2 * w * HD + 18 * w + 4 * w + w + 2 * case["heads"]), "flops": 7.0 * b * w * HD}
    return {"bytes": 2 * _weight_bytes(case["fmt"], case["rows"], case["cols"]), "flops": 0}


def tolerance(case):
    """Four times what the passes below differ by from the 64-bit results on this card, in
    32-bit arithmetic; a step's rounding travels through its layers, and its history codes
    are whole numbers that may fall on the other side of a tie."""
    kind = case["kind"]
    if kind == "pack":
        return "exact"
    if kind == "step":
        return {"rel": 1e-5, "max": 1e-3, "differ": 1e-3}
    if kind == "lm_head":
        return {"rel": 4e-6, "max": 4e-5, "differ": 0.0}
    return {"rel": 4e-6, "max": 1e-4}


# ------------------------------------------------------- the same in 64 bits ----
def _f16(b):
    return b.contiguous().view(torch.float16).double()


def _dequant(fmt, raw, n_values):
    """[rows, n_values] float64 values of rows of K-quant superblocks (or float rows)."""
    rows = raw.shape[0]
    if fmt not in BLOCK:
        return raw.contiguous().view({"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}[fmt]).double()
    blk = raw.reshape(-1, BLOCK[fmt])
    n = blk.shape[0]
    if fmt == "q4k":
        d, dmin, sb, q = _f16(blk[:, 0:2]), _f16(blk[:, 2:4]), blk[:, 4:16].int(), blk[:, 16:144].view(n, 4, 32)
        sc = torch.cat([sb[:, 0:4] & 63, (sb[:, 8:12] & 15) | (sb[:, 0:4] >> 6) << 4], 1).double()
        mn = torch.cat([sb[:, 4:8] & 63, (sb[:, 8:12] >> 4) | (sb[:, 4:8] >> 6) << 4], 1).double()
        code = torch.stack([q & 15, q >> 4], 2).view(n, 8, 32)
        v = code.double() * (d * sc).unsqueeze(2) - (dmin * mn).unsqueeze(2)
    else:
        ql, qh = blk[:, 0:128].view(n, 2, 2, 32).int(), blk[:, 128:192].view(n, 2, 32).int()
        sc, d = blk[:, 192:208].contiguous().view(torch.int8).double(), _f16(blk[:, 208:210])
        low = torch.stack([ql[:, :, 0] & 15, ql[:, :, 1] & 15, ql[:, :, 0] >> 4, ql[:, :, 1] >> 4], 2)
        high = torch.stack([(qh >> s) & 3 for s in (0, 2, 4, 6)], 2)
        v = ((low | high << 4) - 32).double().view(n, 16, 16) * (d * sc).unsqueeze(2)
    return v.reshape(rows, -1)[:, :n_values]


def _product(fmt, raw, cols, x):
    """x W^T in float64, by blocks of rows."""
    return torch.cat([x @ _dequant(fmt, raw[r:r + 8192], cols).t() for r in range(0, raw.shape[0], 8192)], 1)


def _silu(x):
    return x * torch.sigmoid(x)


def _attention64(q, packets, fmt_k, fmt_v, hkv, gate=None, new=None):
    """One sequence: q [hq, hd], packets [positions, bytes] (any order: the softmax is over
    all), new: (k, v) rows of one more position.  Returns out, m, z."""
    kvw, hq = hkv * HD, q.shape[0]
    nb = (kvw + 255) // 256
    split = nb * BLOCK[fmt_k]
    k = _dequant(fmt_k, packets[:, :split], kvw)
    v = _dequant(fmt_v, packets[:, split:split + nb * BLOCK[fmt_v]], kvw)
    if new is not None:
        k, v = torch.cat([k, new[0][None]]), torch.cat([v, new[1][None]])
    s = q.view(hkv, hq // hkv, HD) @ k.view(-1, hkv, HD).permute(1, 2, 0).contiguous() / math.sqrt(HD)
    m = s.amax(-1)
    p = torch.exp(s - m.unsqueeze(-1))
    z = p.sum(-1)
    o = (p @ v.view(-1, hkv, HD).permute(1, 0, 2).contiguous() / z.unsqueeze(-1)).view(hq, HD)
    return (o if gate is None else o * torch.sigmoid(gate)), m.view(hq), z.view(hq)


def _code(x, lo, hi):
    return torch.round(x).clamp(lo, hi)


def _history_values(k, v):
    """Key and value rows after their trip through a history packet (Q4_K, Q6_K)."""
    f16 = lambda x: x.half().double()  # noqa: E731
    x = torch.nn.functional.pad(k, (0, -k.shape[1] % 256)).view(k.shape[0], -1, 8, 32)
    lo, hi = x.amin(-1).clamp(max=0), x.amax(-1).clamp(min=0)
    scale, low = (hi - lo) / 15, -lo
    d, dm = f16(scale.amax(-1, True) / 63), f16(low.amax(-1, True) / 63)
    sc, mn = _code(scale / d.clamp(min=1e-30), 0, 63), _code(low / dm.clamp(min=1e-30), 0, 63)
    code = _code((x + (dm * mn).unsqueeze(-1)) / (d * sc).clamp(min=1e-30).unsqueeze(-1), 0, 15)
    kq = (code * (d * sc).unsqueeze(-1) - (dm * mn).unsqueeze(-1)).reshape(k.shape[0], -1)[:, :k.shape[1]]
    x = torch.nn.functional.pad(v, (0, -v.shape[1] % 256)).view(v.shape[0], -1, 16, 16)
    scale = x.abs().amax(-1) / 31
    d = f16(scale.amax(-1, True) / 127)
    sc = _code(scale / d.clamp(min=1e-30), 0, 127)
    code = _code(x / (d * sc).clamp(min=1e-30).unsqueeze(-1), -32, 31)
    return kq, (code * (d * sc).unsqueeze(-1)).reshape(v.shape[0], -1)[:, :v.shape[1]]


def _delta64(raw, conv, taps, a, b, a_log, dt_bias, state, norm, gate):
    """One token of a delta-net layer: (gated output, conv window, state) in float64."""
    batch, heads = a.shape
    w = heads * HD
    window = torch.cat([conv, raw.unsqueeze(-1)], -1)
    y = _silu((window * taps).sum(-1)).view(batch, 3, heads, HD)
    q, k = (t / torch.sqrt((t * t).sum(-1, True) + 1e-6) for t in (y[:, 0], y[:, 1]))
    decay = torch.exp(-torch.exp(a_log) * torch.nn.functional.softplus(a + dt_bias))
    state = state * decay[..., None, None]
    err = torch.sigmoid(b).unsqueeze(-1) * (y[:, 2] - (state * k.unsqueeze(2)).sum(-1))
    state = state + err.unsqueeze(-1) * k.unsqueeze(2)
    o = (state * q.unsqueeze(2)).sum(-1) / math.sqrt(HD)
    o = o / torch.sqrt((o * o).mean(-1, True) + 1e-6) * norm.view(heads, HD) * _silu(gate.view(batch, heads, HD))
    return o.view(batch, w), window[..., 1:], state


def _step64(case, seed):
    m = _decode_model(case, seed, False, keep=True)
    mat = lambda n: torch.as_tensor(m.gguf[n], device=DEV)  # noqa: E731
    vec = lambda n: torch.as_tensor(m.gguf[n], device=DEV).double()  # noqa: E731
    hq, hkv, h, hid, batch = case["q_heads"], case["kv_heads"], case["rec_heads"], case["hidden"], case["batch"]
    s, ctx = h * HD, _contexts(case, batch)
    rms = lambda x, w: x / torch.sqrt((x * x).mean(-1, True) + 1e-6) * w  # noqa: E731
    packets, rec, conv = _state_part(m, "packets"), _state_part(m, "recurrent"), _state_part(m, "conv")
    x = _dequant("q4k", m.embed[m.tokens.long()], hid)
    pos = torch.tensor(ctx, device=DEV).double()
    phase = pos[:, None] * 1e6 ** (-torch.arange(HD // 2, device=DEV).double() / (HD // 2))
    cos, sin = phase.cos()[:, None], phase.sin()[:, None]

    def rotate(t):
        a, b = t[..., 0::2], t[..., 1::2]
        return torch.stack([a * cos - b * sin, a * sin + b * cos], -1).reshape(t.shape)

    lf = lr = 0
    states, windows = [], []
    for l in range(case["layers"]):
        n = rms(x, vec(f"{l}.norm_in"))
        p = _product("q4k", mat(f"{l}.w_in"), hid, n)
        if l % 4 == 3:
            q = rotate(rms(p[:, :hq * HD].reshape(batch, hq, HD), vec(f"{l}.q_norm").view(hq, HD)))
            k = rotate(rms(p[:, hq * HD:(hq + hkv) * HD].reshape(batch, hkv, HD), vec(f"{l}.k_norm").view(hkv, HD)))
            kq, vq = _history_values(k.reshape(batch, -1), p[:, (hq + hkv) * HD:])
            o = torch.stack([_attention64(q[i], packets[lf, i, :ctx[i]], "q4k", "q6k", hkv, new=(kq[i], vq[i]))[0]
                             for i in range(batch)]).view(batch, -1)
            lf += 1
        else:
            o, cw, st = _delta64(p[:, :3 * s], conv[lr].double(), vec(f"{l}.conv_w"), p[:, 4 * s:4 * s + h],
                                 p[:, 4 * s + h:], vec(f"{l}.a_log"), vec(f"{l}.dt_bias"), rec[lr].double(),
                                 vec(f"{l}.out_norm"), p[:, 3 * s:4 * s])
            states.append(st)
            windows.append(cw)
            lr += 1
        x = x + _product("q4k", mat(f"{l}.w_o"), o.shape[1], o)
        n = rms(x, vec(f"{l}.norm_post"))
        act = _silu(_product("q4k", mat(f"{l}.w_gate"), hid, n)) * _product("q4k", mat(f"{l}.w_up"), hid, n)
        x = x + _product("q4k", mat(f"{l}.w_down"), case["ff"], act)
    logits = _product("q6k", mat("lm_head"), hid, rms(x, vec("norm_final")))
    return dict(logits=logits, tokens=None, recurrent=torch.stack(states), conv=torch.stack(windows), packets=None)


def exact(case, seed):
    kind = case["kind"]
    if kind == "pack":
        return None   # bytes
    if kind == "step":
        return _step64(case, seed)
    s = prepare(case, seed)
    if kind == "gemv":
        y = _product(case["fmt"], s["raw"], case["cols"], s["x"].double())
        return y + s["y"].double() if case["accumulate"] else y
    if kind == "mlp":
        x = s["x"].double()
        act = _silu(_product("q4k", s["raw"][0], case["hidden"], x)) * _product("q4k", s["raw"][1], case["hidden"], x)
        y = _product(case["fmt_d"], s["raw"][2], case["inter"], act)
        return act, y + s["y"].double() if case["accumulate"] else y
    if kind == "lm_head":
        return _product(case["fmt"], s["raw"], case["hidden"], s["h"].double()), None
    if kind == "attention":
        got = []
        base, ctx = s["base"].tolist(), s["ctx"].tolist()
        for i in range(case["nseq"]):
            used = min(ctx[i], case["capacity"])
            got.append(_attention64(s["q"][i].double(), s["packets"][base[i]:base[i] + used], case["fmt_k"],
                                    case["fmt_v"], case["hkv"], None if s["gate"] is None else s["gate"][i].double()))
        return tuple(torch.stack(t) for t in zip(*got))
    h = case["heads"]
    w = h * HD
    p = s["proj"].double()
    out, conv, state = _delta64(p[:, :3 * w], s["conv"].double(), s["taps"].double(), p[:, 4 * w:4 * w + h],
                                p[:, 4 * w + h:], s["a_log"].double(), s["dt_bias"].double(), s["state"].double(),
                                s["norm"].double(), p[:, 3 * w:4 * w])
    return dict(out=out, conv=conv, state=state)
