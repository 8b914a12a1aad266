"""GPU: sessions opened on a closed session's memory (the context keeps it for
the next one). A session that takes over the blocks of a larger, a smaller or an
equal one, with other sessions open beside it, gives the bits that a session on
fresh memory gives: prompt logits, greedy tokens and state."""
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
