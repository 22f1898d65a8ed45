"""Batched prefill of models with K-quant / F32 matrices against their own decode runs (which
test_kquant_engine_gpu.py and test_kquant_proj_gpu.py pin to the oracle): every position's h_nextn, the last
token's logits, the KV cache and the recurrent state bit for bit, at lengths around the 32-token matrix tiles and
the 64-token workgroup tiles and at lengths whose launches take four waves per workgroup, and the MTP rows seeded in
one pass. The layers hold every K-quant type in every role, F32 and K-quant beta / alpha, split and interleaved
gate / up, K-quant and Q8_0 down. Blocks and activations of the largest integers that the formats hold go through
every type's products."""
import os

import numpy as np
import pytest

import gguf_writer as W
import kquant_blocks as KB
import oracle as O
from test_prefill_gpu import assert_same_state, bits, decode, prompt

pytestmark = pytest.mark.gpu

T = O.T
Q3, Q4, Q5, Q6, F32 = 11, 12, 13, 14, 0


def model_types(variant):
    roles = {  # layer -> (mixer projection parts, output, gate, up, down, shared gate, up, down)
        0: ([Q4] * 4, Q4, Q3, Q3, Q3, Q6, Q6, Q6),
        1: ([Q5, Q6, F32, F32], Q5, Q4, Q5, Q6, 8, 8, Q4),
        2: ([8, 8, F32, F32], 8, Q4, Q4, Q5, Q3, Q5, 8),
        3: ([Q4, Q6, Q3], Q6, Q6, Q6, 8, 8, 8, 8),
        4: ([Q6, Q4, Q5], Q3, 8, 8, Q4, Q4, Q4, Q5),
    }
    if variant == "one type a layer":
        roles = {0: ([Q3] * 4, Q5, Q3, Q3, Q3, Q4, Q4, Q6), 1: ([Q5] * 4, Q6, Q5, Q5, Q5, Q6, Q6, Q3),
                 2: ([Q6] * 4, Q3, Q6, Q6, Q6, Q3, Q3, Q5), 3: ([Q4] * 3, Q4, Q4, Q4, Q4, Q5, Q5, Q4)}
    if variant == "q8_0 mixers":
        roles = {0: ([8, 8, F32, F32], Q4, Q4, Q4, Q5, 8, 8, 8), 3: ([8, 8, 8], 8, 8, 8, 8, Q5, Q5, Q3),
                 4: ([8, 8, 8], 8, Q4, Q4, Q5, 8, 8, 8)}
    ty = {}
    for layer, (proj, out, *moe) in roles.items():
        att = layer in (3, 4)
        kinds = ("ATT_Q", "ATT_K", "ATT_V") if att else ("DN_QKV", "DN_Z", "DN_BETA", "DN_ALPHA")
        names = kinds + ("ATT_OUT" if att else "DN_OUT", "GATE_EXPS", "UP_EXPS", "DOWN_EXPS", "GATE_SHEXP", "UP_SHEXP",
                         "DOWN_SHEXP")
        for name, t in zip(names, (*proj, out, *moe)):
            if t != 8:
                ty[(layer, T[name])] = t
    ty[(O.GLOBAL_LAYER, T["OUTPUT"])] = Q6
    if variant != "q8_0 mixers":
        ty[(O.GLOBAL_LAYER, T["TOK_EMBD"])] = Q4
    return ty


@pytest.mark.parametrize("variant", ["every type", "q8_0 mixers"])
@pytest.mark.parametrize("n", [3, 9, 31, 33, 64, 65, 150])
def test_typed_prefill_equals_decode(variant, n):
    typed_prefill_equals_decode(variant, n, 256)


@pytest.mark.parametrize("n,second", [(475, 9), (2059, 3)])
def test_typed_prefill_in_wide_workgroups_equals_decode(n, second):
    """Prompts whose launches have enough tiles for four waves per workgroup, with two 32-token tiles and with one:
    475 tokens for the projections (the last token tile has 18, and the waves past the 32 beta / alpha rows none), 2048
    (then a second chunk) for every plain launch but the shared gate / up, and with 64 pairs per expert"""
    typed_prefill_equals_decode("one type a layer", n, 2304, second)


def typed_prefill_equals_decode(variant, n, n_ctx, second=None):
    import oxe_amd as A
    d = O.desc_small()
    ty = model_types(variant)
    a, b = (A.Engine(d, seed=7, n_ctx=n_ctx, types=ty) for _ in range(2))
    toks = prompt(d, n)
    print(f"typed prefill {variant} n={n}", flush=True)
    second = second or n // 3
    for lo, hi in ((0, n - second), (n - second, n)):   # a second prompt continues the first
        nx, h = a.prefill(toks[lo:hi], hidden=True)
        x, hs = decode(b, toks[lo:hi])
        assert nx == x
        assert np.array_equal(bits(h), bits(hs)), f"rows {sorted(set(np.nonzero(bits(h) != bits(hs))[0]))[:8]}"
        assert np.array_equal(bits(a.hidden(0)), bits(b.hidden(0)))
        assert np.array_equal(bits(a.logits(0)), bits(b.logits(0)))
        assert_same_state(a, b, d, f"{variant} {lo}..{hi}")
    for _ in range(3):
        nx, x = a.step(nx), b.step(x)
        assert nx == x
        assert np.array_equal(bits(a.logits(0)), bits(b.logits(0)))
    for e in (a, b):
        e.close()


@pytest.mark.parametrize("variant", ["every type", "q8_0 mixers"])
def test_typed_seeding_equals_seeding_runs(variant):
    import oxe_amd as A
    d = O.desc_small()
    a, b = (A.Engine(d, seed=7, n_ctx=256, types=model_types(variant)) for _ in range(2))
    toks = prompt(d, 75)
    print(f"typed MTP prefill {variant}", flush=True)
    x = a.mtp_prefill_batched(toks)
    assert x == b.mtp_prefill(toks)
    for i in range(4):
        got, want = a.mtp_step(x), b.mtp_step(x)
        assert got == want, i
        x = want[-1]
    assert np.array_equal(bits(a.hidden(0)), bits(b.hidden(0)))
    for name, ka, kb in zip(("K", "V^T"), *[[e.state(w, 2 * 2 * 256 * 256 * 2, dtype=np.uint16) for w in (0, 1)] for e in (a, b)]):
        assert np.array_equal(ka, kb), name
    for e in (a, b):
        e.close()


def extreme_blocks(ty, rows, k):
    """rows of random blocks with the block's largest integers in three rows of four: scale * code and min at their
    largest, their largest without mins (or the largest of the other sign), and the same against the codes' other end"""
    w = KB.random_blocks(ty, rows, k, seed=90 + ty, d_range=(1e-5, 2e-5), dw=None).reshape(rows, -1, KB.BYTES[ty])
    if ty in (4, 5):
        w[0::4, :, 4:] = 255                        # scales 63, mins 63, codes 15 / 31
        w[1::4, :, 4:] = 255
        w[1::4, :, 8:12] = 0                        # mins 0
        w[1::4, :, 12:16] = 0x0F
        w[2::4, :, 4:16] = 255                      # largest scales and mins, random codes
    elif ty == 3:
        w[0::4, :, :108] = 0                        # scale -32, code -4
        w[1::4, :, :108] = 255                      # scale 31, code 3
        w[2::4, :, :96], w[2::4, :, 96:108] = 0, 255   # scale 31, code -4
    else:
        w[0::4, :, :192], w[0::4, :, 192:208] = 0, 128      # scale -128, code -32
        w[1::4, :, :192], w[1::4, :, 192:208] = 255, 127    # scale 127, code 31
        w[2::4, :, :192], w[2::4, :, 192:208] = 255, 128    # scale -128, code 31
    return np.ascontiguousarray(w)


def test_typed_prefill_of_extreme_blocks_equals_decode():
    """A model whose residual stream stays the token's embedding (every other matrix is zero), of one magnitude and any
    signs: the q8_K codes are all -127, all 127 or mixed signs of 127, their sums of 16 up to 2032. Its delta-net layers'
    qkv are extreme blocks of one type each; the conv state holds their last three rows of outputs as they are."""
    import oxe_amd as A
    d = O.desc_small(n_layer=5, full_attention_interval=5, n_vocab=256)
    E, qkv = d.n_embd, {0: 3, 1: 4, 2: 5, 3: 6}
    ty = {(il, T["DN_QKV"]): t + 8 for il, t in qkv.items()}
    ty.update({(il, T[k]): Q6 for il in qkv for k in ("DN_Z", "DN_BETA", "DN_ALPHA")})
    ty.update({(il, T[f"{k}_EXPS"]): Q3 for il in range(6) for k in ("GATE", "UP", "DOWN")})
    rng = np.random.default_rng(5)
    codes = np.full((256, E), 127, np.int8)
    codes[1::4] = -127
    codes[2::4] = rng.choice(np.array([-127, 127], np.int8), (64, E))
    codes[3::4] = np.repeat(rng.choice(np.array([-127, 127], np.int8), (64, E // 16)), 16, axis=1)
    scales = np.repeat(rng.uniform(1e-3, 2e-3, (256, 1)).astype(np.float16).view(np.uint16), E // 32, axis=1)
    tensors = []
    for name, t, shape, payload in W.synth_model_tensors(O, d, 3, ty):
        if name == "token_embd.weight":
            payload = W.q8_blocks(codes, scales)
        elif name.endswith(".attn_norm.weight"):
            payload = np.ones(E, np.float32).tobytes()
        elif name.endswith("attn_qkv.weight"):
            payload = extreme_blocks(t - 8, shape[1], E).tobytes()
        elif t != F32:
            payload = lambda f, n=W.tensor_bytes(t, shape): f.seek(n, os.SEEK_CUR)   # noqa: E731
        tensors.append((name, t, shape, payload))
    base = "/dev/shm" if os.path.isdir("/dev/shm") and os.access("/dev/shm", os.W_OK) else "/tmp"
    path = os.path.join(base, f"oxe_test_kqx_{os.getpid()}.gguf")
    try:
        print("writing the model of extreme blocks", flush=True)
        W.write(path, W.qwen35moe_meta(d), tensors)
        a, b = (A.Engine.from_gguf(path, n_ctx=768) for _ in range(2))
    finally:
        if os.path.exists(path):
            os.remove(path)
    at = 0
    for n, kinds in ((4, (0, 1, 2)), (5, (3, 0, 3)), (35, (2, 1, 0)), (66, (0, 2, 1)), (460, (1, 3, 0))):
        toks = [int(v) for v in rng.integers(0, 256, n)]
        toks[-3:] = [4 * (t // 4) + k for t, k in zip(toks[-3:], kinds)]   # the last three tokens' outputs are compared
        print(f"extreme blocks, {n} tokens at {at}", flush=True)
        a.prefill(toks)
        decode(b, toks)
        assert_same_state(a, b, d, f"{n} tokens at {at}", main_only=True)
        conv = a.state(2, 4 * 8192 * 3 * 4, dtype=np.float32)
        assert np.isfinite(conv).all() and (np.abs(conv) > 0).mean() > 0.99
        at += n
    for e in (a, b):
        e.close()
