"""Batched prefill of models with K-quant / F32 matrices against their own decode runs (which
test_kquant_engine_gpu.py and test_kquant_proj_gpu.py pin to the oracle): every position's h_nextn, the last
token's logits, the KV cache and the recurrent state bit for bit, at lengths around the 32-token matrix tiles and
the 64-token workgroup tiles, and the MTP rows seeded in one pass. The layers hold every K-quant type in
every role, F32 and K-quant beta / alpha, split and interleaved gate / up, K-quant and Q8_0 down."""
import numpy as np
import pytest

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
@pytest.mark.parametrize("n", [3, 31, 33, 64, 65, 150])
def test_typed_prefill_equals_decode(variant, n):
    import oxe_amd as A
    d = O.desc_small()
    ty = model_types(variant)
    a, b = (A.Engine(d, seed=7, n_ctx=256, types=ty) for _ in range(2))
    toks = prompt(d, n)
    print(f"typed prefill {variant} n={n}", flush=True)
    for lo, hi in ((0, n - n // 3), (n - n // 3, n)):   # a second prompt continues the first
        nx, h = a.prefill(toks[lo:hi], hidden=True)
        x, hs = decode(b, toks[lo:hi])
        assert nx == x
        assert np.array_equal(bits(h), bits(hs)), f"rows {sorted(set(np.nonzero(bits(h) != bits(hs))[0]))[:8]}"
        assert np.array_equal(bits(a.hidden(0)), bits(b.hidden(0)))
        assert np.array_equal(bits(a.logits(0)), bits(b.logits(0)))
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
