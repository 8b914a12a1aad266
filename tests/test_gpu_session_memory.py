"""GPU: sessions opened on a closed session's memory (the context keeps it for
the next one). A session that takes over the blocks of a larger, a smaller or an
equal one, with other sessions open beside it, gives the bits that a session on
fresh memory gives: prompt logits, greedy tokens and state. What the context
keeps is one session's memory however many were opened in turn, and
Context.trim gives it back."""
import ctypes as C

import numpy as np
import pytest

import clibs
import ornithology_amd as oa

pytestmark = pytest.mark.gpu


def request(m, prompt, gen):
    s = m.session(len(prompt) + gen)
    s.eval(prompt)
    first = s.logits().copy()
    return s, (first, s.generate(gen), s.logits().copy(), s.delta_state(0).copy(), *s.kv(3))


def test_sessions_on_reused_memory(monkeypatch):
    monkeypatch.setenv("ORNITH_PREFILL_SERIAL", "0")
    rng = np.random.default_rng(5)
    prompts = [rng.integers(0, clibs.C1["vocab"], n).astype(np.int32) for n in (300, 1, 77, 301, 200, 64, 290)]
    want = []
    for p in prompts:                     # each on a context of its own: fresh memory
        ctx = oa.Context(0)
        m = ctx.synth(**clibs.C1)
        s, r = request(m, p, 5)
        want.append(r)
        s.free()
        m.free()
        ctx.close()
    ctx = oa.Context(0)
    m = ctx.synth(**clibs.C1)
    held = None
    for _ in range(2):
        for k, p in enumerate(prompts):
            s, got = request(m, p, 5)
            for a, b in zip(got, want[k]):
                assert np.array_equal(a.view(np.uint8), b.view(np.uint8)), k
            if held is not None:
                held.free()
            held = s                      # one session stays open beside the next
    held.free()
    m.free()
    ctx.close()


def test_closed_sessions_memory_serves_the_next():
    ctx = oa.Context(0)
    m = ctx.synth(**clibs.C1)
    p = np.random.default_rng(6).integers(0, clibs.C1["vocab"], 500).astype(np.int32)

    def kept(caps, n=500):
        for cap in caps:
            s = m.session(cap)
            s.eval(p[:n])
            s.free()
        return ctx.trim()

    kept([4000])
    one = kept([4000])
    assert one > 4000 * 2 * (64 + 4)          # the KV codes and scales of one KV head at least
    assert ctx.trim() == 0
    assert kept([4000] * 6) == one            # each took the one before it's
    assert kept([4000, 3500, 3900, 4000]) == one
    assert kept([4000, 64000]) > one          # too small for the next: both are kept
    a, b = m.session(4000), m.session(4000)   # open together: no memory in common
    a.eval(p)
    b.eval(p)
    a.free()
    b.free()
    assert kept([4000]) == 2 * one - 4000 * 32 * 8   # the RoPE table is the model's
    x = clibs.gauss(8, "kept", 256 * 4096)
    ctx.quantize(clibs.Q4_K, x)
    enc = ctx.trim()
    assert enc >= x.nbytes
    for _ in range(3):
        ctx.quantize(clibs.Q4_K, x)
    assert ctx.trim() == enc
    kept([4000])
    m.free()                                  # gives back what its sessions held
    assert ctx.trim() == 0
    m = ctx.synth(**clibs.C1)
    m.session(4000).free()
    m.free()
    assert ctx.trim() == 0
    ctx.close()


def test_rope_tables_go_with_their_sessions():
    """A table that a longer session's outgrew goes with the last session that
    reads it, the longest with Context.trim; a session that still reads one goes on."""
    L = oa.lib()

    def free_bytes():
        f, t = C.c_size_t(), C.c_size_t()
        assert L.hipMemGetInfo(C.byref(f), C.byref(t)) == 0
        return f.value

    ctx = oa.Context(0)
    m = ctx.synth(**clibs.C1)
    p = np.random.default_rng(7).integers(0, clibs.C1["vocab"], 40).astype(np.int32)
    first = m.session(60)
    first.eval(p)
    want, tokens = first.logits().copy(), first.generate(9)
    first.free()
    ctx.trim()
    start = free_bytes()
    table = 32 * 8                            # bytes of a position: pairs of a head of 64
    short = m.session(400_000)
    s = m.session(900_000)                    # a table of its own; short's was the model's
    ctx.trim()
    both = free_bytes()
    short.eval(p)
    assert np.array_equal(short.logits().view(np.uint32), want.view(np.uint32))
    assert np.array_equal(short.generate(9), tokens)
    short.free()
    ctx.trim()
    # its KV cache, scores and table; half of the table's size of slack
    least = 400_000 * (2 * 2 * (64 + 4) + 8 * 4 + table)
    assert free_bytes() - both > least - 200_000 * table
    s.free()
    ctx.trim()
    assert free_bytes() > start - (16 << 20)
    s = m.session(60)
    s.eval(p)
    assert np.array_equal(s.logits().view(np.uint32), want.view(np.uint32))
    s.free()
    m.free()
    ctx.close()
