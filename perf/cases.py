"""The work that a program built on this library has it do, as cases that can be timed and compared.

Every case goes through the public entry points (include/llamd_hip.h, the Python wrappers of llamd_rs_amd.rocm) at the
widths of a Qwen3-30B-A3B layer (2048 hidden, 32 query and 4 kv heads of 128, 128 experts of 768, top 8, 151936
vocabulary), the configuration that this repository's benchmark and tests use, over the batch sizes, prompt lengths and
contexts that serving meets. Weights are N(0, 0.05) values quantized to Q6_K, activations N(0, 1).

  attn_in   RMSNorm, Q8_K and the Q/K/V projections of 1..16 sequences
  attend    attention over the KV cache for 1..16 sequences of 32..8192 positions, and the Q8_K of its output
  moe       one MoE layer for 1..32 sequences behind a handle: router, top 8, experts, combine, residual
  moe_ffi   the same FFN as the reference's device model queues it, call by call, weights in its planar form
  prefill   the grouped expert FFN of 24..2048 prompt tokens, bit-exact or within the reduction tolerance
  head      the LM head of 1..16 sequences: logits and arg-max
  linear    the f32 matrix product of the tensor Backend, for layers kept in F32
  model     one token of a whole (two-layer) model at a position of its context
"""
import math
import os
import tempfile

import numpy as np
import torch

from llamd_rs_amd import ffi_replay, gguf_writer, rocm
from llamd_rs_amd._lib import lib
from llamd_rs_amd.gguf import Gguf

EMBD, HEADS, KV_HEADS, HEAD_DIM = 2048, 32, 4, 128
FF, EXPERTS, USED, VOCAB = 768, 128, 8, 151936
EPS, ROPE_BASE = 1e-6, 1e6
SIGMA = 0.05
DEV = "cuda"


# ---- the cases -----------------------------------------------------------------

def listed():
    return [
        # the front end of one decode step for one user: two short launches, the smallest call there is
        {"name": "attn_in_1", "kind": "attn_in", "nseq": 1},
        # one user deep in a long conversation: every step reads the whole cache
        {"name": "attend_1_4100", "kind": "attend", "nseq": 1, "ctx": 4100, "heads": 32, "kv_heads": 4, "hd": 128},
        # a batch of users at different lengths of ordinary conversations
        {"name": "attend_13_1000", "kind": "attend", "nseq": 13, "ctx": 1000, "heads": 32, "kv_heads": 4, "hd": 128},
        # the FFN of one decode step for one user, most of a token's time
        {"name": "moe_1", "kind": "moe", "nseq": 1},
        # the same for a full decode batch: most experts are touched
        {"name": "moe_16", "kind": "moe", "nseq": 16},
        # a caller of the reference's own FFI with a few sequences in flight
        {"name": "moe_ffi_6", "kind": "moe_ffi", "nseq": 6},
        # a short prompt: as many experts as tokens, few tokens for each
        {"name": "prefill_45", "kind": "prefill", "n_tok": 45, "skew": 1.1, "reduction": False},
        # the benchmark's prompt chunk with its skewed routing
        {"name": "prefill_512", "kind": "prefill", "n_tok": 512, "skew": 1.1, "reduction": False},
        # a long prompt, evenly routed, by a caller that takes the reduction tolerance
        {"name": "prefill_2000_red", "kind": "prefill", "n_tok": 2000, "skew": 0.6, "reduction": True},
        # the vocabulary projection of a full decode batch
        {"name": "head_16", "kind": "head", "nseq": 16, "rows": VOCAB, "reduction": False},
        # an unquantized projection over a prompt through the tensor Backend
        {"name": "linear_200", "kind": "linear", "m": 2048, "n": 200, "k": 2048},
        # the whole call: one token through two layers and the head, mid-conversation
        {"name": "model_700", "kind": "model", "pos": 700},
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    kind = rng.choice(["attn_in", "attend", "attend", "moe", "moe_ffi", "prefill", "prefill", "head", "linear", "model"])
    if kind in ("attn_in", "moe_ffi"):
        return {"kind": kind, "nseq": _log(rng, 1, 16)}
    if kind == "moe":
        return {"kind": kind, "nseq": _log(rng, 1, 32)}
    if kind == "attend":
        nseq = _log(rng, 1, 16)
        heads, kv_heads, hd = rng.choice([(32, 4, 128), (32, 4, 128), (16, 8, 128), (12, 12, 64)])
        return {"kind": kind, "nseq": nseq, "ctx": _log(rng, 32, min(8192, 32768 // nseq)), "heads": heads,
                "kv_heads": kv_heads, "hd": hd}
    if kind == "prefill":
        return {"kind": kind, "n_tok": _log(rng, 24, 2000), "skew": rng.choice([0.0, 0.6, 1.1]),
                "reduction": rng.random() < 0.5}
    if kind == "head":
        return {"kind": kind, "nseq": _log(rng, 1, 16), "rows": rng.choice([32003, VOCAB]),
                "reduction": rng.random() < 0.3}
    if kind == "linear":
        return {"kind": kind, "m": _log(rng, 100, 2048), "n": _log(rng, 1, 200), "k": _log(rng, 128, 2048)}
    return {"kind": kind, "pos": _log(rng, 20, 1200)}


# ---- inputs ----------------------------------------------------------------------

def _gen(seed, stream):
    return torch.Generator(device=DEV).manual_seed(seed * 64 + stream)


def _normal(seed, stream, *shape, sigma=1.0):
    return torch.randn(*shape, generator=_gen(seed, stream), device=DEV) * sigma


def _q6k_codes(seed, stream, rows, k):
    """(codes [n][256] 0..63, scales [n][16], d [n] f16) of rows x k weights ~ N(0, SIGMA), by 256-value block; the
    scale of each 16 is its largest magnitude over 32, as Q6_K quantizers choose it."""
    x = _normal(seed, stream, rows * k // 256, 16, 16, sigma=SIGMA)
    top = x.abs().amax(-1)
    d = (top.amax(-1, keepdim=True) / (127 * 32)).half()
    sc = (top / 32 / d.float()).round().clamp(1, 127)
    x.div_((d.float() * sc)[..., None]).round_().add_(32).clamp_(0, 63)
    return x.to(torch.uint8).reshape(-1, 256), sc.to(torch.int8), d.reshape(-1)


def _q6k_bytes(seed, stream, rows, k):
    """The ggml bytes of that matrix, on the host."""
    q, sc, d = _q6k_codes(seed, stream, rows, k)
    n = q.shape[0]
    q = q.reshape(n, 2, 4, 32)
    out = torch.empty(n, 210, dtype=torch.uint8, device=DEV)
    out[:, :128] = ((q[:, :, :2] & 15) | ((q[:, :, 2:] & 15) << 4)).reshape(n, 128)
    hi = q >> 4
    out[:, 128:192] = (hi[:, :, 0] | (hi[:, :, 1] << 2) | (hi[:, :, 2] << 4) | (hi[:, :, 3] << 6)).reshape(n, 64)
    out[:, 192:208] = sc.view(torch.uint8)
    out[:, 208:210] = d[:, None].view(torch.uint8)
    return out.reshape(-1).cpu().numpy()


def _q6k_values(seed, stream, rows, k):
    """The same matrix dequantized, in 64 bits."""
    q, sc, d = _q6k_codes(seed, stream, rows, k)
    w = (q.double() - 32).reshape(-1, 16, 16) * (d.double()[:, None] * sc.double())[..., None]
    return w.reshape(rows, k)


def _weights(seed, stream, rows, k):
    return rocm.DeviceWeights.upload(_q6k_bytes(seed, stream, rows, k), rows, k // 256)


def _experts():
    return (("gate", 1, FF, EMBD), ("up", 2, FF, EMBD), ("down", 3, EMBD, FF))


def _router(seed):
    return _normal(seed, 0, EXPERTS, EMBD, sigma=0.02)


def _moe_layer(seed):
    w = {name: _q6k_bytes(seed, s, EXPERTS * rows, k) for name, s, rows, k in _experts()}
    return rocm.MoeLayer(_router(seed).cpu().numpy(), w["gate"], w["up"], w["down"], EMBD, FF, EXPERTS, USED)


def _popularity(skew):
    p = torch.arange(1, EXPERTS + 1, dtype=torch.float64) ** -skew
    return p / p.sum()


def _routing(seed, n_tok, skew):
    """Top-8 ids and renormalised weights of n_tok tokens, expert popularity a power law in a shuffled order."""
    g = _gen(seed, 7)
    p = _popularity(skew).to(DEV)[torch.randperm(EXPERTS, generator=g, device=DEV)]
    u = torch.rand(n_tok, EXPERTS, generator=g, device=DEV, dtype=torch.float64).clamp_min(1e-12)
    ids = (p.log() - (-u.log()).log()).topk(USED).indices.int().contiguous()
    w = torch.rand(n_tok, USED, generator=g, device=DEV).sort(descending=True).values + 0.05
    return ids, (w / w.sum(-1, keepdim=True)).contiguous()


def _lengths(case):
    """Positions in the cache of each sequence: from all of ctx down to half of it."""
    n, ctx = case["nseq"], case["ctx"]
    return [max(1, ctx - s * ctx // (2 * n)) for s in range(n)]


def _empty(*shape, dtype=torch.float32):
    return torch.empty(*shape, dtype=dtype, device=DEV)


def _write_model(path, seed, layers):
    """A GGUF of the layer widths above; the layers share one copy of their tensors' bytes."""
    kv = KV_HEADS * HEAD_DIM
    near_one = lambda s, n: (1 + 0.1 * _normal(seed, s, n)).cpu().numpy()  # noqa: E731
    layer = {
        "attn_norm.weight": ([EMBD], near_one(11, EMBD)),
        "ffn_norm.weight": ([EMBD], near_one(12, EMBD)),
        "attn_q_norm.weight": ([HEAD_DIM], near_one(13, HEAD_DIM)),
        "attn_k_norm.weight": ([HEAD_DIM], near_one(14, HEAD_DIM)),
        "attn_q.weight": ([EMBD, HEADS * HEAD_DIM], _q6k_bytes(seed, 15, HEADS * HEAD_DIM, EMBD)),
        "attn_k.weight": ([EMBD, kv], _q6k_bytes(seed, 16, kv, EMBD)),
        "attn_v.weight": ([EMBD, kv], _q6k_bytes(seed, 17, kv, EMBD)),
        "attn_output.weight": ([HEADS * HEAD_DIM, EMBD], _q6k_bytes(seed, 18, EMBD, HEADS * HEAD_DIM)),
        "ffn_gate_inp.weight": ([EMBD, EXPERTS], _router(seed).cpu().numpy()),
    }
    for name, s, rows, k in _experts():
        layer["ffn_%s_exps.weight" % name] = ([k, rows, EXPERTS], _q6k_bytes(seed, s, EXPERTS * rows, k))
    tensors = {
        "token_embd.weight": ([EMBD, VOCAB], _q6k_bytes(seed, 19, VOCAB, EMBD)),
        "output.weight": ([EMBD, VOCAB], _q6k_bytes(seed, 20, VOCAB, EMBD)),
        "output_norm.weight": ([EMBD], near_one(21, EMBD)),
    }
    for i in range(layers):
        tensors.update({"blk.%d.%s" % (i, n): t for n, t in layer.items()})
    u32, f32, arch = gguf_writer.U32, gguf_writer.F32, "qwen3moe"
    meta = [("general.architecture", gguf_writer.STRING, arch), (arch + ".block_count", u32, layers),
            (arch + ".embedding_length", u32, EMBD), (arch + ".attention.head_count", u32, HEADS),
            (arch + ".attention.head_count_kv", u32, KV_HEADS), (arch + ".attention.key_length", u32, HEAD_DIM),
            (arch + ".attention.layer_norm_rms_epsilon", f32, EPS), (arch + ".rope.freq_base", f32, ROPE_BASE),
            (arch + ".expert_count", u32, EXPERTS), (arch + ".expert_used_count", u32, USED),
            (arch + ".expert_feed_forward_length", u32, FF), (arch + ".feed_forward_length", u32, 6144),
            (arch + ".context_length", u32, 40960)]
    gguf_writer.write(path, meta, [(n, d, 0 if a.dtype == np.float32 else 14, a) for n, (d, a) in tensors.items()])


def prepare(case, seed):
    L, kind, n = lib(), case["kind"], case.get("nseq", 1)
    if L.llamd_fwd_stream_init():
        raise RuntimeError("no stream")
    s = {"case": case}
    if kind == "attn_in":
        rows = (HEADS * HEAD_DIM, KV_HEADS * HEAD_DIM, KV_HEADS * HEAD_DIM)
        s.update(w=[_weights(seed, i + 1, r, EMBD) for i, r in enumerate(rows)], rows=rows,
                 x=_normal(seed, 8, n, EMBD), norm=1 + _normal(seed, 9, EMBD, sigma=0.1), aq=_empty(n, EMBD, dtype=torch.int8),
                 ad=_empty(n, EMBD // 256), xn=_empty(n, EMBD), inv=_empty(n), out=[_empty(n, r) for r in rows])
    elif kind == "attend":
        heads, kvh, hd = case["heads"], case["kv_heads"], case["hd"]
        max_kv = -(-case["ctx"] // 256) * 256
        meta = torch.tensor([[1, t - 1] for t in _lengths(case)], dtype=torch.int32, device=DEV)
        s.update(q=_normal(seed, 1, n, heads * hd), kc=_normal(seed, 2, n, max_kv, kvh * hd),
                 vc=_normal(seed, 3, n, max_kv, kvh * hd), meta=meta, max_kv=max_kv, out=_empty(n, heads * hd),
                 scores=_empty(n, heads * max_kv), aq=_empty(n, heads * hd, dtype=torch.int8),
                 ad=_empty(n, heads * hd // 256))
    elif kind == "moe":
        s.update(layer=_moe_layer(seed), x=_normal(seed, 8, n, EMBD), res=_normal(seed, 9, n, EMBD), out=_empty(n, EMBD))
    elif kind == "moe_ffi":
        for name, st, rows, k in _experts():
            data, off = ffi_replay.planar_repack(_q6k_bytes(seed, st, EXPERTS * rows, k), EXPERTS * rows, k // 256)
            s[name] = (rocm.DeviceBuffer.from_array(data), off)
        s.update(router=_router(seed), x=_normal(seed, 8, n, EMBD), norm=1 + _normal(seed, 9, EMBD, sigma=0.1),
                 xn=_empty(n, EMBD), inv=_empty(n), logits=_empty(n, EXPERTS), probs=_empty(n, EXPERTS),
                 ids=_empty(n, USED, dtype=torch.int32), weights=_empty(n, USED), gate_out=_empty(n, USED * FF),
                 up_out=_empty(n, USED * FF), act=_empty(n, USED * FF), down_out=_empty(n, USED * EMBD),
                 aq=_empty(n, USED * FF, dtype=torch.int8), sums=_empty(n, USED * FF // 16, dtype=torch.int32),
                 ad=_empty(n, USED * FF // 256), out=_empty(n, EMBD))
    elif kind == "prefill":
        ids, w = _routing(seed, case["n_tok"], case["skew"])
        s.update(layer=_moe_layer(seed), x=_normal(seed, 8, case["n_tok"], EMBD), ids=ids, weights=w,
                 out=_empty(case["n_tok"], EMBD))
    elif kind == "head":
        s.update(head=rocm.LmHead(_weights(seed, 1, case["rows"], EMBD), max_seq=n), x=_normal(seed, 8, n, EMBD),
                 logits=_empty(n, case["rows"]), ids=_empty(n, dtype=torch.int32))
    elif kind == "linear":
        s.update(w=_normal(seed, 1, case["m"], case["k"], sigma=SIGMA), x=_normal(seed, 2, case["n"], case["k"]),
                 out=_empty(case["n"], case["m"]))
    else:
        fd, path = tempfile.mkstemp(suffix=".gguf")
        os.close(fd)
        try:
            _write_model(path, seed, 2)
            with Gguf(path) as g:
                s["model"] = rocm.DeviceModel(g, max_kv=2048)
        finally:
            os.unlink(path)
        tokens = torch.randint(VOCAB, (case["pos"] + 1,), generator=_gen(seed, 30), device=DEV).tolist()
        for pos, t in enumerate(tokens[:-1]):
            s["model"].forward(t, pos)
        s["token"] = tokens[-1]
    torch.cuda.synchronize()
    return s


# ---- one pass ----------------------------------------------------------------------

def _moe_ffi(L, s, n):
    p = {k: v.data_ptr() for k, v in s.items() if isinstance(v, torch.Tensor)}
    (gate, fg), (up, fu), (down, fd) = ((s[k][0].ptr, s[k][1]) for k in ("gate", "up", "down"))
    eb, fb = EMBD // 256, FF // 256
    if n == 1:
        L.llamd_fwd_rms_norm_quant(p["x"], p["norm"], p["xn"], p["aq"], p["ad"], p["inv"], EMBD, EPS)
        L.llamd_fwd_matvec_f32(p["router"], p["xn"], p["logits"], EMBD, EXPERTS)
        L.llamd_fwd_router(p["logits"], EXPERTS, USED, p["ids"], p["weights"], p["probs"])
        L.llamd_fwd_planar_grouped_x2(gate, fg, up, fu, p["ids"], p["aq"], p["ad"], p["gate_out"], p["up_out"], eb, FF, USED)
        L.llamd_fwd_silu_mul(p["gate_out"], p["up_out"], p["act"], USED * FF)
        L.llamd_fwd_quantize(p["act"], p["aq"], p["ad"], USED * fb)
        L.llamd_fwd_planar_grouped_pa(down, fd, p["ids"], p["aq"], p["ad"], p["down_out"], fb, EMBD, USED)
        L.llamd_fwd_moe_combine_add(p["down_out"], p["weights"], p["x"], p["out"], USED, EMBD)
    else:
        L.llamd_u_norm_quant(p["x"], p["norm"], p["xn"], p["aq"], p["sums"], p["ad"], p["inv"], EMBD, n, EPS)
        L.llamd_b_matvec_f32(p["router"], p["xn"], p["logits"], EMBD, EXPERTS, n)
        L.llamd_b_router(p["logits"], EXPERTS, USED, p["ids"], p["weights"], p["probs"], n)
        L.llamd_u_grouped_x2(gate, fg, up, fu, p["ids"], p["aq"], p["sums"], p["ad"], p["gate_out"], p["up_out"], eb, FF,
                             USED, n)
        L.llamd_b_silu_mul(p["gate_out"], p["up_out"], p["act"], USED * FF * n)
        L.llamd_u_quantize(p["act"], p["aq"], p["sums"], p["ad"], USED * fb * n)
        L.llamd_u_grouped_pa(down, fd, p["ids"], p["aq"], p["sums"], p["ad"], p["down_out"], fb, EMBD, USED, n)
        L.llamd_b_moe_combine_add(p["down_out"], p["weights"], p["x"], p["out"], USED, EMBD, n)
    return {"out": s["out"], "ids": s["ids"], "weights": s["weights"]}


def run(state):
    s, case, L = state, state["case"], lib()
    kind, n = case["kind"], case.get("nseq", 1)
    rc = 0
    if kind == "attn_in":
        x, w, xn, aq, ad, inv = (s[k].data_ptr() for k in ("x", "norm", "xn", "aq", "ad", "inv"))
        m, o = [t.ptr for t in s["w"]], [t.data_ptr() for t in s["out"]]
        if n == 1:
            L.llamd_fwd_rms_norm_quant(x, w, xn, aq, ad, inv, EMBD, EPS)
            L.llamd_fwd_matvec_x3(*m, aq, ad, *o, EMBD // 256, *s["rows"])
        else:
            L.llamd_b_rms_norm_quant(x, w, xn, aq, ad, inv, EMBD, n, EPS)
            L.llamd_b_matvec_x3(*m, aq, ad, *o, EMBD // 256, *s["rows"], n)
        return s["out"]
    if kind == "attend":
        q, kc, vc, out, sc, meta, aq, ad = (s[k].data_ptr() for k in ("q", "kc", "vc", "out", "scores", "meta", "aq", "ad"))
        heads, kvh, hd = case["heads"], case["kv_heads"], case["hd"]
        if n == 1:
            L.llamd_fwd_attention_meta(q, kc, vc, out, sc, heads, kvh, hd, meta, s["max_kv"])
            L.llamd_fwd_quantize(out, aq, ad, heads * hd // 256)
        else:
            L.llamd_b_attention(q, kc, vc, out, sc, heads, kvh, hd, s["max_kv"], meta, n)
            L.llamd_b_quantize(out, aq, ad, n * heads * hd // 256)
        return {"out": s["out"], "quants": s["aq"], "scales": s["ad"]}
    if kind == "moe":
        x, res, out = (s[k].data_ptr() for k in ("x", "res", "out"))
        if n == 1:
            rc = L.llamd_hip_moe_forward(s["layer"].handle, x, res, out, 0)
        else:
            rc = L.llamd_hip_moe_forward_batch(s["layer"].handle, x, res, out, n)
        result = s["out"]
    elif kind == "moe_ffi":
        result = _moe_ffi(L, s, n)
    elif kind == "prefill":
        rc = L.llamd_hip_moe_prefill_ex(s["layer"].handle, s["x"].data_ptr(), s["ids"].data_ptr(), s["weights"].data_ptr(),
                                        s["out"].data_ptr(), case["n_tok"], 1 if case["reduction"] else 0)
        result = s["out"]
    elif kind == "head":
        rc = L.llamd_hip_lmhead_forward_ex(s["head"].handle, s["x"].data_ptr(), n, s["logits"].data_ptr(),
                                           s["ids"].data_ptr(), 1 if case["reduction"] else 0)
        result = {"logits": s["logits"], "ids": s["ids"]}
    elif kind == "linear":
        rc = L.llamd_hip_be_matmul(s["w"].data_ptr(), s["x"].data_ptr(), s["out"].data_ptr(), case["m"], case["n"], case["k"])
        result = s["out"]
    else:
        logits, token = s["model"].forward(s["token"], case["pos"])
        result = {"logits": logits, "token": token}
    if rc:
        raise RuntimeError("%s: %s" % (kind, L.llamd_hip_last_error()))
    return result


# ---- what a pass cannot do without -----------------------------------------------------

def _q6k(rows, k):
    return rows * k // 256 * 210


def _moe_work(tokens, touched):
    pair = 2 * 3 * FF * EMBD  # multiply-adds of one expert on one token, as operations
    return touched * 3 * _q6k(FF, EMBD) + tokens * EMBD * 8, tokens * USED * pair


def _touched(tokens, skew):
    p = _popularity(skew)
    return float((1 - (1 - p.clamp(max=1 / USED) * USED).clamp(min=0) ** tokens).sum())


def work(case):
    kind, n = case["kind"], case.get("nseq", 1)
    kv = KV_HEADS * HEAD_DIM
    if kind == "attn_in":
        rows = HEADS * HEAD_DIM + 2 * kv
        return {"bytes": _q6k(rows, EMBD) + 4 * n * (EMBD + rows), "flops": 2 * n * rows * EMBD}
    if kind == "attend":
        t, q = sum(_lengths(case)), case["heads"] * case["hd"]
        return {"bytes": 8 * t * case["kv_heads"] * case["hd"] + n * q * 9, "flops": 4 * t * q}
    if kind in ("moe", "moe_ffi"):
        b, f = _moe_work(n, _touched(n, 0.0))
        return {"bytes": b + 4 * EXPERTS * EMBD, "flops": f + 2 * n * EXPERTS * EMBD}
    if kind == "prefill":
        b, f = _moe_work(case["n_tok"], _touched(case["n_tok"], case["skew"]))
        return {"bytes": b, "flops": f}
    if kind == "head":
        return {"bytes": _q6k(case["rows"], EMBD) + 4 * n * (EMBD + case["rows"]), "flops": 2 * n * case["rows"] * EMBD}
    if kind == "linear":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": 4 * (m * k + n * k + m * n), "flops": 2 * m * n * k}
    b, f = _moe_work(1, USED)
    attn = _q6k(2 * HEADS * HEAD_DIM + 2 * kv, EMBD) + 8 * (case["pos"] + 1) * kv
    return {"bytes": 2 * (b + 4 * EXPERTS * EMBD + attn) + _q6k(VOCAB, EMBD) + 4 * VOCAB,
            "flops": 2 * (f + 2 * EMBD * (2 * HEADS * HEAD_DIM + 2 * kv) + 4 * (case["pos"] + 1) * HEADS * HEAD_DIM)
            + 2 * EMBD * VOCAB}


def tolerance(case):
    # every entry point but the reduction ones promises the reference CPU path's bits (its operations in its order)
    if not case.get("reduction"):
        return "exact"
    if case["kind"] == "head":
        # one f32 rounding a block instead of eight: 1e-7 and 5.3e-7 from the bit-exact logits; ids are certified
        return {"rel": 5e-7, "max": 3e-6}
    # the SwiGLU outputs are rounded to 8 bits between the two products, and now and then one falls to the next value:
    # 5.7e-5 and 3.8e-3 from the bit-exact outputs
    return {"rel": 2.5e-4, "max": 1.6e-2}


# ---- the same in 64 bits ------------------------------------------------------------------

def _q8k(x):
    """The rows of x after rounding to Q8_K (256-value blocks of 8-bit codes and an f32 scale), in 64 bits."""
    b = x.float().reshape(-1, 256)
    top = b.gather(1, b.abs().argmax(1, keepdim=True))
    inverse = -127.0 / top
    q = (inverse * b).round().clamp(max=127)
    return torch.where(top == 0, 0.0, q.double() * (1.0 / inverse).double()).reshape(x.shape)


def _norm(x, w):
    x = x.double()
    return x / (x.square().mean(-1, keepdim=True) + EPS).sqrt() * w.double()


def _ffn(seed, x, ids, weights):
    """sum over the routed experts of weight * down(silu(gate x) * up x), x already in f32."""
    values = {name: _q6k_values(seed, s, EXPERTS * rows, k).reshape(EXPERTS, rows, k) for name, s, rows, k in _experts()}
    xq, out = _q8k(x), torch.zeros(x.shape, dtype=torch.float64, device=DEV)
    for e in range(EXPERTS):
        at, slot = (ids == e).nonzero(as_tuple=True)
        if len(at):
            g, u = xq[at] @ values["gate"][e].T, xq[at] @ values["up"][e].T
            act = _q8k(g / (1 + (-g).exp()) * u)
            out.index_add_(0, at, weights.double()[at, slot, None] * (act @ values["down"][e].T))
    return out


def _route(seed, x):
    p = torch.softmax(x.double() @ _router(seed).double().T, -1)
    top = p.topk(USED)
    return top.indices, top.values / top.values.sum(-1, keepdim=True)


def exact(case, seed):
    kind, n = case["kind"], case.get("nseq", 1)
    if kind == "attn_in":
        x = _q8k(_norm(_normal(seed, 8, n, EMBD), 1 + _normal(seed, 9, EMBD, sigma=0.1)))
        rows = (HEADS * HEAD_DIM, KV_HEADS * HEAD_DIM, KV_HEADS * HEAD_DIM)
        return [x @ _q6k_values(seed, i + 1, r, EMBD).T for i, r in enumerate(rows)]
    if kind == "attend":
        heads, kvh, hd = case["heads"], case["kv_heads"], case["hd"]
        max_kv = -(-case["ctx"] // 256) * 256
        q = _normal(seed, 1, n, heads * hd).double().reshape(n, heads, 1, hd)
        k, v = (_normal(seed, i, n, max_kv, kvh * hd) for i in (2, 3))
        out = []
        for s, t in enumerate(_lengths(case)):
            ks, vs = (c[s, :t].double().reshape(t, kvh, hd).transpose(0, 1).repeat_interleave(heads // kvh, 0).contiguous()
                      for c in (k, v))
            p = torch.softmax(q[s] @ ks.transpose(1, 2).contiguous() / math.sqrt(hd), -1)
            out.append((p @ vs).reshape(-1))
        return {"out": torch.stack(out), "quants": None, "scales": None}
    if kind == "moe":
        x = _normal(seed, 8, n, EMBD)
        return _normal(seed, 9, n, EMBD).double() + _ffn(seed, x, *_route(seed, x))
    if kind == "moe_ffi":
        x = _normal(seed, 8, n, EMBD)
        xn = _norm(x, 1 + _normal(seed, 9, EMBD, sigma=0.1))
        ids, w = _route(seed, xn)
        return {"out": x.double() + _ffn(seed, xn, ids, w), "ids": None, "weights": w}
    if kind == "prefill":
        return _ffn(seed, _normal(seed, 8, case["n_tok"], EMBD), *_routing(seed, case["n_tok"], case["skew"]))
    if kind == "head":
        return {"logits": _q8k(_normal(seed, 8, n, EMBD)) @ _q6k_values(seed, 1, case["rows"], EMBD).T, "ids": None}
    if kind == "linear":
        return _normal(seed, 2, case["n"], case["k"]).double() @ _normal(seed, 1, case["m"], case["k"], sigma=SIGMA).double().T
    return None  # a whole model's cache in 64 bits would take minutes
