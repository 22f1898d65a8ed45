"""Device memory of the batched prefill: what its buffers hold as prompts grow, and what happens when they do
not fit. The engine's own limit (oxe_engine_limit_bytes) stands in for a full device."""
import numpy as np
import pytest

import oracle as O
from test_kquant_prefill_gpu import model_types
from test_prefill_gpu import assert_same_state, bits, prompt

pytestmark = pytest.mark.gpu


def held(e):
    import oxe_amd as A
    return A.lib().oxe_engine_device_bytes(e.h)


def limit(e, n):
    import oxe_amd as A
    A.lib().oxe_engine_limit_bytes(e.h, n)


def test_typed_prefill_without_memory_runs_as_decode():
    """a typed engine prefills and seeds without the buffers, bit for bit as with them, and takes them
    once there is room"""
    import oxe_amd as A
    d = O.desc_small()
    a, b = (A.Engine(d, seed=7, n_ctx=256, types=model_types("every type")) for _ in range(2))
    before = held(a)
    limit(a, before)
    toks = prompt(d, 75)
    print("typed MTP prefill, no memory for its buffers", flush=True)
    x = a.mtp_prefill_batched(toks[:32])
    assert x == b.mtp_prefill_batched(toks[:32])
    for _ in range(3):
        got, want = a.mtp_step(x), b.mtp_step(x)
        assert got == want
        x = want[-1]
    assert_same_state(a, b, d, "after MTP steps")
    print("typed prefill, no memory for its buffers", flush=True)
    for lo, hi in ((32, 65), (65, 75)):
        (x, hx), (y, hy) = a.prefill(toks[lo:hi], hidden=True), b.prefill(toks[lo:hi], hidden=True)
        assert x == y and a.pos == b.pos
        assert np.array_equal(bits(hx), bits(hy))
        assert np.array_equal(bits(a.logits(0)), bits(b.logits(0)))
        assert np.array_equal(bits(a.hidden(0)), bits(b.hidden(0)))
        assert_same_state(a, b, d, f"{lo}..{hi}")
    assert held(a) == before
    limit(a, 0)
    assert a.prefill(toks[:20]) == b.prefill(toks[:20])
    assert held(a) > before
    assert_same_state(a, b, d, "with the buffers")
    for e in (a, b):
        e.close()


def test_q8_0_prefill_without_memory_is_refused():
    """an all-Q8_0 engine says so and stays usable"""
    import oxe_amd as A
    d = O.desc_small()
    a, b = (A.Engine(d, seed=7, n_ctx=256) for _ in range(2))
    toks = prompt(d, 40)
    limit(a, held(a))
    with pytest.raises(RuntimeError, match="out of device memory for the prefill buffers"):
        a.prefill(toks)
    assert a.pos == 0
    assert a.step(toks[0]) == b.step(toks[0])
    limit(a, 0)
    assert a.prefill(toks) == b.prefill(toks)
    assert_same_state(a, b, d, "after the limit went")
    for e in (a, b):
        e.close()


@pytest.mark.parametrize("types", [None, "every type"])
def test_growing_prompts_hold_one_set_of_buffers(types):
    """a longer prompt's buffers replace the shorter one's; a set that does not fit leaves none behind"""
    import oxe_amd as A
    d = O.desc_small()
    ty = types and model_types(types)
    a, b = (A.Engine(d, seed=7, n_ctx=512, types=ty) for _ in range(2))
    toks = prompt(d, 240)
    bare = held(b)
    b.prefill(toks[:100])
    for lo, hi in ((0, 20), (20, 60), (60, 140), (140, 240)):   # 20, 40, 80, 100 tokens
        print(f"prefill {types} {lo}..{hi}", flush=True)
        x = a.prefill(toks[lo:hi])
    assert held(a) == held(b) > bare
    b.prefill(toks[100:190])
    assert x == b.prefill(toks[190:])
    assert held(a) == held(b)
    assert_same_state(a, b, d, "grown against one size", main_only=True)
    limit(a, held(a))
    print(f"prefill {types} at the limit", flush=True)
    if ty:
        assert a.prefill(toks[:120]) == b.prefill(toks[:120])
    else:
        with pytest.raises(RuntimeError, match="out of device memory"):
            a.prefill(toks[:120])
        b.prefill(toks[:120])
        for t in toks[:120]:
            a.step(t)
    assert held(a) == bare
    assert a.prefill(toks[:50]) == b.prefill(toks[:50])   # what fits is taken again
    assert held(a) > bare
    for e in (a, b):
        e.close()
