"""The work that is timed when this engine is made faster: what its users have it do.

Two kinds of user. A program that brings its own model calls the kernel-level products (the lane
GEMVs of a decode step, the GEMM of a prompt, over Q8_0 or K-quant weights). A server holds an engine
with a whole 35B-A3B-shaped model, all Q8_0 or with the matrix types of the Ornith or Qwen3.6 files,
takes prompts in and generates tokens with MTP speculation. Sizes are the model's, the benchmark's
(config 1's 4096 x 2048 matrix, the 2048-token prompt, 512 prior positions) or generic.

Every path's contract (include/oxe_amd.h) is the reference's result bit for bit: per output one fp32
chain in a fixed order over exact integer block sums. So another correct implementation shows no
difference at all, and the tolerance of every case is "exact".
"""
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "snapdragon-engine_amd"))
import oxe_amd as A  # noqa: E402

DEV = "cuda"
VOCAB = {"q8_0": 151936, "ornith": 248320, "qwen36": 248320}
KQ_BYTES = {3: 110, 4: 144, 5: 176, 6: 210}   # bytes of a 256-weight block of Q3_K .. Q6_K


# ---- the cases -------------------------------------------------------------------------------------

def listed():
    return [
        # one projection of a verify step: two tokens' activations through a 4096 x 2048 matrix
        dict(name="gemv_two_lanes", op="gemv", k=2048, nr=4096, nl=2),
        # the LM head for one token: the largest single product of a decode step
        dict(name="gemv_head", op="gemv", k=2048, nr=151936, nl=1),
        # a model of another width: a row length without round numbers, ragged rows, three lanes
        dict(name="gemv_odd_width", op="gemv", k=1120, nr=3001, nl=3),
        # the Ornith file's delta-net projection of a verify step
        dict(name="kgemv_projection", op="kgemv", ty=4, k=2048, nr=8192, nl=2),
        # both files' LM head of a verify step
        dict(name="kgemv_head", op="kgemv", ty=6, k=2048, nr=248320, nl=2),
        # a long prompt through a delta-net projection: float activations in, float rows out
        dict(name="gemm_prompt", op="gemm", k=2048, nr=12352, nt=2048),
        # a short chat turn through an output projection, fewer tokens than a tile
        dict(name="gemm_short_turn", op="gemm", k=4096, nr=2048, nt=45),
        # a server's greedy generation after a cached prefix, all Q8_0
        dict(name="decode_q8_0", op="decode", types="q8_0", layers=40, prefix=512, steps=4),
        # the same with the matrix types of a file that mixes Q8_0, K-quant and F32 matrices
        dict(name="decode_qwen36", op="decode", types="qwen36", layers=40, prefix=65, steps=4),
        # a long prompt into an empty context, whole model, MTP rows seeded
        dict(name="prefill_q8_0", op="prefill", types="q8_0", layers=40, prefix=0, tokens=2048),
        # the next turn of a chat: a short prompt after a cached prefix
        dict(name="prefill_q8_0_turn", op="prefill", types="q8_0", layers=40, prefix=700, tokens=61),
        # a prompt into a stack of layers with the Ornith file's types, every position's hidden state
        dict(name="prefill_ornith", op="prefill", types="ornith", layers=8, prefix=0, tokens=701),
    ]


def _log(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    op = rng.choice(["gemv", "gemv", "kgemv", "kgemv", "gemm", "gemm", "decode", "prefill", "prefill"])
    if op == "gemv":
        k = rng.choice([512, 2048, 4096, 32 * _log(rng, 10, 160), 32 * _log(rng, 10, 160)])
        return dict(op=op, k=k, nr=_log(rng, 700, min(151936, 151936 * 2048 // k)), nl=rng.randint(1, 4))
    if op == "kgemv":
        ty, k = rng.choice([3, 4, 5, 6]), 256 * rng.choice([2, 4, 8, 8, 12, 16])
        return dict(op=op, ty=ty, k=k, nr=_log(rng, 500, min(248320, 248320 * 2048 // k)), nl=rng.randint(1, 4))
    if op == "gemm":
        k = rng.choice([512, 2048, 4096, 128 * _log(rng, 5, 40)])
        return dict(op=op, k=k, nr=_log(rng, 500, min(12352, 12352 * 2048 // k)), nt=_log(rng, 9, 2048))
    types = rng.choice(["q8_0", "ornith", "qwen36"])
    if op == "decode":
        return dict(op=op, types=types, layers=rng.choice([4, 8, 20]),
                    prefix=_log(rng, 9, 1500) if types == "q8_0" else _log(rng, 9, 90), steps=rng.randint(2, 5))
    layers = rng.choice([4, 8])
    if types == "q8_0":
        return dict(op=op, types=types, layers=layers, prefix=rng.choice([0, _log(rng, 20, 900)]),
                    tokens=_log(rng, 11, 2048))
    return dict(op=op, types=types, layers=layers, prefix=0, tokens=_log(rng, 11, 5600 // layers))


def tolerance(case):
    return "exact"


# ---- inputs ----------------------------------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed * 7919 + 17)


def _normal(g, *shape):
    return torch.randn(*shape, generator=g, device=DEV)


def _q8_0(x):
    """Q8_0 blocks of float rows: codes int8, scales fp16 (bits in int16)."""
    b = x.view(*x.shape[:-1], -1, 32)
    d = b.abs().amax(-1) / 127.0
    inv = torch.where(d != 0, 1.0 / d, torch.zeros_like(d))
    q = torch.round(b * inv[..., None]).to(torch.int8).view(x.shape)
    return q, d.to(torch.float16).view(torch.int16)


def _q8_0_weights(g, nr, k):
    """Rows of a matrix as a quantised model holds them, made in pieces."""
    q = torch.empty((nr, k), dtype=torch.int8, device=DEV)
    d = torch.empty((nr, k // 32), dtype=torch.int16, device=DEV)
    for r in range(0, nr, 16384):
        q[r:r + 16384], d[r:r + 16384] = _q8_0(_normal(g, min(16384, nr - r), k) * k ** -0.5)
    return q, d


def _q8_K(x):
    """ggml block_q8_K bytes of float rows: f32 scale, 256 codes, 16 sums of 16."""
    b = x.view(x.shape[0], -1, 256)
    at = b.abs().argmax(-1, keepdim=True)
    inv = -127.0 / torch.gather(b, -1, at)
    q = torch.round(b * inv).clamp(-128, 127).to(torch.int8)
    sums = q.view(*q.shape[:-1], 16, 16).to(torch.int32).sum(-1).to(torch.int16)
    parts = (1.0 / inv).contiguous().view(torch.uint8), q.view(torch.uint8), sums.contiguous().view(torch.uint8)
    return torch.cat(parts, -1).reshape(x.shape[0], -1).contiguous()


def _f16_at(blocks, at, value):
    blocks[:, at:at + 2] = value.to(torch.float16).view(torch.uint8).view(-1, 2)


def _kq_weights(g, ty, nr, k):
    """K-quant rows: random codes and sub-block scales, block scales of a model's size."""
    n = nr * (k // 256)
    b = torch.randint(0, 256, (n, KQ_BYTES[ty]), dtype=torch.uint8, device=DEV, generator=g)
    scale = (torch.rand(n, device=DEV, generator=g) + 0.5) * k ** -0.5 / 256
    if ty in (4, 5):
        _f16_at(b, 0, scale)
        _f16_at(b, 2, scale * 7)
    else:
        _f16_at(b, KQ_BYTES[ty] - 2, scale)
    return b.view(nr, -1)


def _types(kind, layers):
    """Matrix types of the named file's layers for a stack of `layers` (the file's 40 as they are)."""
    if kind == "q8_0":
        return None
    q3, q4, q5, q6, f32 = (A._TYPE_ID[t] for t in ("Q3_K", "Q4_K", "Q5_K", "Q6_K", "F32"))
    n, t = A._MATRIX_KIND, {(63, A._GLOBAL_KIND["output.weight"]): q6}
    edge = max(1, layers // 8)
    if kind == "ornith":
        t[(63, A._GLOBAL_KIND["token_embd.weight"])] = q4
    for il in range(layers + 1):
        mtp = il == layers
        if kind == "qwen36":
            for name in ("gate", "up"):
                t[(il, n[f"ffn_{name}_exps.weight"])] = q4
            t[(il, n["ffn_down_exps.weight"])] = q6 if il in (layers - 6, layers - 2, layers - 1) else q5
            if not mtp and (il + 1) % 4:
                t[(il, n["ssm_beta.weight"])] = t[(il, n["ssm_alpha.weight"])] = f32
        elif not mtp:
            mixer = (("attn_qkv", "attn_gate", "ssm_beta", "ssm_alpha", "ssm_out") if (il + 1) % 4
                     else ("attn_q", "attn_k", "attn_v", "attn_output"))
            for name in mixer:
                t[(il, n[f"{name}.weight"])] = q4
            for name in ("gate", "up", "down"):
                t[(il, n[f"ffn_{name}_exps.weight"])] = q4 if il < edge or il >= layers - edge else q3
                t[(il, n[f"ffn_{name}_shexp.weight"])] = q6
    return t


def _engine(case, seed, n_ctx):
    kind, layers = case["types"], case["layers"]
    return A.Engine(A.desc_35b_a3b(n_layer=layers, n_vocab=VOCAB[kind]), seed=seed, n_ctx=n_ctx,
                    types=_types(kind, layers))


def prepare(case, seed):
    op = case["op"]
    if op in ("decode", "prefill"):
        rng = np.random.RandomState(seed % 2 ** 31)
        n_new = case["tokens"] if op == "prefill" else 2 * case["steps"] + 2
        e = _engine(case, seed, case["prefix"] + n_new + 8)
        ids = rng.randint(1000, 151000, case["prefix"] + n_new).astype(np.uint32)
        s = dict(case=case, e=e, srv=A.ServerEngine(e, mtp=op == "decode" or case["types"] == "q8_0"))
        if case["prefix"]:
            s["x"] = e.mtp_prefill_batched(ids[:case["prefix"]])
            s["snap"] = s["srv"].snapshot()   # a server's cached prefix
        s["new"] = ids[case["prefix"]:]
        return s
    g = _gen(seed)
    if op == "kgemv":
        return dict(case=case, w=_kq_weights(g, case["ty"], case["nr"], case["k"]),
                    x=_q8_K(_normal(g, case["nl"], case["k"])))
    w = _q8_0_weights(g, case["nr"], case["k"])
    if op == "gemv":
        return dict(case=case, w=w, x=_q8_0(_normal(g, case["nl"], case["k"])))
    return dict(case=case, w=w, x=_normal(g, case["nt"], case["k"]))


# ---- one pass --------------------------------------------------------------------------------------

def run(s):
    case = s["case"]
    op = case["op"]
    if op == "gemv":
        return A.gemv_q8_0(*s["w"], *s["x"])
    if op == "kgemv":
        return A.vl_gemv(case["ty"], s["w"], case["k"], s["x"])
    if op == "gemm":   # a linear layer over a prompt: the activations quantised, then the product
        return A.gemm_q8_0(*s["w"], *A.quantize_q8_0(s["x"]))
    e, srv = s["e"], s["srv"]
    if op == "decode":
        srv.restore(s["snap"])
        cap = 2 * case["steps"] + 2
        e.mtp_device_begin(s["x"], cap)
        e.mtp_device_steps(case["steps"])
        toks, nxt = e.mtp_device_end(cap)
        return np.array(toks, np.int64), nxt, e.logits(0)
    if case["prefix"]:
        srv.restore(s["snap"])
    else:
        srv.reset()
    if case["types"] == "q8_0":
        return srv.prefill(s["new"])
    return e.prefill(s["new"], hidden=True)


# ---- what a pass cannot do without -----------------------------------------------------------------

# bits per weight of each matrix type, block scales included
_BITS = {8: 8.5, 0: 32.0, 11: 110 / 32, 12: 144 / 32, 13: 176 / 32, 14: 210 / 32}
E, FF, EXPERTS, USED = 2048, 512, 256, 8


def _stack(case):
    """(bytes outside the experts, bytes of one expert summed over layers, weights per token) of the
    layers, and the same three of the MTP layer and of the LM head."""
    t, layers = _types(case["types"], case["layers"]) or {}, case["layers"]
    n = A._MATRIX_KIND
    dn = {"attn_qkv": 8192 * E, "attn_gate": 4096 * E, "ssm_beta": 32 * E, "ssm_alpha": 32 * E, "ssm_out": 4096 * E}
    at = {"attn_q": 8192 * E, "attn_k": 512 * E, "attn_v": 512 * E, "attn_output": 4096 * E}
    got = []
    for ils in (range(layers), [layers]):
        dense = exp = macs = 0.0
        for il in ils:
            bits = lambda name: _BITS[t.get((il, n[name + ".weight"]), 8)]  # noqa: E731
            mixer = dn if il < layers and (il + 1) % 4 else at
            shared = {f"ffn_{m}_shexp": FF * E for m in ("gate", "up", "down")}
            extra = {"nextn.eh_proj": 2 * E * E} if il == layers else {}
            for name, w in {**mixer, **shared, **extra}.items():
                dense += w * bits(name) / 8
                macs += w
            dense += (EXPERTS + 1) * E * 4
            macs += (EXPERTS + 1) * E + 3 * USED * FF * E
            exp += sum(FF * E * bits(f"ffn_{m}_exps") / 8 for m in ("gate", "up", "down"))
        got += [dense, exp, macs]
    head = VOCAB[case["types"]] * E
    return got + [head * _BITS[t.get((63, A._GLOBAL_KIND["output.weight"]), 8)] / 8, head]


def work(case):
    op = case["op"]
    if op == "gemv":
        k, nr, nl = case["k"], case["nr"], case["nl"]
        return dict(bytes=nr * k * 34 / 32 + nl * k * 34 / 32 + nl * nr * 4, flops=2 * nl * nr * k)
    if op == "kgemv":
        k, nr, nl = case["k"], case["nr"], case["nl"]
        return dict(bytes=nr * (k // 256) * KQ_BYTES[case["ty"]] + nl * (k // 256) * 292 + nl * nr * 4,
                    flops=2 * nl * nr * k)
    if op == "gemm":
        k, nr, nt = case["k"], case["nr"], case["nt"]
        return dict(bytes=nr * k * 34 / 32 + nt * k * 4 + nt * nr * 4, flops=2 * nt * nr * k)
    dense, exp, macs, m_dense, m_exp, m_macs, head, h_macs = _stack(case)
    n_att, pos = case["layers"] // 4, case["prefix"]
    n_dn, kv, state = case["layers"] - n_att, 2048, 2 * 2 ** 20 + 98304
    if op == "decode":   # per step: a draft, then a verify of two tokens (their experts' union)
        union = EXPERTS * (1 - (1 - USED / EXPERTS) ** 2)
        step = (dense + exp * union + head + 3 * n_dn * state + n_att * pos * kv
                + m_dense + m_exp * USED + head + pos * kv)
        return dict(bytes=case["steps"] * step,
                    flops=case["steps"] * 2 * (2 * (macs + h_macs) + m_macs + h_macs))
    nt = case["tokens"]
    union = EXPERTS * (1 - (1 - USED / EXPERTS) ** nt)
    att = n_att * 16 * 256 * 2 * sum(pos + i + 1 for i in range(nt))   # scores and values
    rule = n_dn * nt * 32 * 128 * 128 * 3
    rows = nt * E * 4 if case["types"] != "q8_0" else 0
    return dict(bytes=dense + exp * union + head + 2 * n_dn * state + n_att * (pos + nt) * kv + rows,
                flops=2 * (nt * macs + h_macs + att + rule))


# ---- the same in 64 bits ---------------------------------------------------------------------------

def _f64_q8_0(q, d):
    b = q.double().view(*q.shape[:-1], -1, 32)
    return (b * d.view(torch.float16).double()[..., None]).view(q.shape)


def _f64_kq(ty, w):
    """Values of K-quant rows [nr, nb * bytes] -> float64 [nr, nb * 256]."""
    b = w.view(-1, KQ_BYTES[ty])
    f16 = lambda at: b[:, at:at + 2].contiguous().view(torch.float16).double()  # noqa: E731
    i = b.to(torch.int32)
    if ty in (4, 5):
        sc = i[:, 4:16]
        lo, hi = torch.cat([sc[:, :4] & 63, (sc[:, 8:] & 15) | (sc[:, :4] >> 6 << 4)], 1), \
            torch.cat([sc[:, 4:8] & 63, (sc[:, 8:] >> 4) | (sc[:, 4:8] >> 6 << 4)], 1)
        qs = i[:, -128:].view(-1, 4, 1, 32)
        q = torch.cat([qs & 15, qs >> 4], 2).view(-1, 8, 32)
        if ty == 5:
            bit = torch.arange(8, device=w.device).view(1, 8, 1)
            q = q + ((i[:, 16:48].view(-1, 1, 32) >> bit & 1) << 4)
        v = (f16(0) * lo)[..., None] * q - (f16(2) * hi)[..., None]
    elif ty == 6:
        ql, qh = i[:, :128].view(-1, 2, 1, 2, 32), i[:, 128:192].view(-1, 2, 1, 32)
        low = torch.cat([ql & 15, ql >> 4], 2).view(-1, 2, 4, 32)
        shift = torch.arange(0, 8, 2, device=w.device).view(1, 1, 4, 1)
        q = (low | (qh >> shift & 3) << 4) - 32
        sc = b[:, 192:208].contiguous().view(torch.int8).double()
        v = (f16(208) * sc)[..., None] * q.view(-1, 16, 16)
    else:
        s = i[:, 96:108]
        raw = torch.cat([s[:, :8] & 15, s[:, :8] >> 4], 1)
        top = torch.cat([s[:, 8:] >> sh & 3 for sh in (0, 2, 4, 6)], 1)
        shift = torch.arange(0, 8, 2, device=w.device).view(1, 1, 4, 1)
        low = (i[:, 32:96].view(-1, 2, 1, 32) >> shift & 3).view(-1, 8, 32)
        bit = torch.arange(8, device=w.device).view(1, 8, 1)
        q = low - 4 + 4 * (i[:, :32].view(-1, 1, 32) >> bit & 1)
        v = (f16(108) * ((raw | top << 4) - 32))[..., None] * q.view(-1, 16, 16)
    return v.reshape(w.shape[0], -1)


def exact(case, seed):
    op = case["op"]
    if op in ("decode", "prefill"):
        return None   # whole engines: the model in 64 bits takes minutes
    s = prepare(case, seed)
    if op == "kgemv":
        y = s["x"].view(case["nl"], -1, 292)
        x = (y[..., 4:260].contiguous().view(torch.int8).double()
             * y[..., :4].contiguous().view(torch.float32).double()).view(case["nl"], -1)
        rows = lambda r: _f64_kq(case["ty"], s["w"][r:r + 8192])  # noqa: E731
    else:
        x = _f64_q8_0(*(s["x"] if op == "gemv" else _q8_0(s["x"])))
        rows = lambda r: _f64_q8_0(s["w"][0][r:r + 8192], s["w"][1][r:r + 8192])  # noqa: E731
    return torch.cat([x @ rows(r).T for r in range(0, case["nr"], 8192)], 1)
