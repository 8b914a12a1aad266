"""GPU: a context, its models and their sessions freed in any order. The last of
them gives the device memory back, and what is freed after the context or the
model does not reach into it."""
import ctypes as C
import itertools

import numpy as np
import pytest

import clibs
import ornithology_amd as oa

pytestmark = pytest.mark.gpu

CFG = dict(clibs.C1, n_layers=2, full_interval=2)


def free_bytes():
    f, t = C.c_size_t(), C.c_size_t()
    assert oa.lib().hipMemGetInfo(C.byref(f), C.byref(t)) == 0
    return f.value


def opened():
    ctx = oa.Context(0)
    m = ctx.synth(**CFG)
    s = m.session(300_000)            # 128 MB and more of session memory
    s.eval(np.arange(40, dtype=np.int32))
    return {"context": ctx.close, "model": m.free, "session": s.free}


def test_free_in_any_order():
    for f in opened().values():       # what the process allocates once is there
        f()
    start = free_bytes()
    for order in itertools.permutations(("context", "model", "session")):
        d = opened()
        assert free_bytes() < start - (100 << 20)
        for k in order:
            d[k]()
        assert free_bytes() > start - (32 << 20), order


def test_other_sessions_go_on():
    """A session whose context handle is closed, and one beside a freed one."""
    ctx = oa.Context(0)
    m = ctx.synth(**CFG)
    p = np.arange(50, dtype=np.int32)
    a, b = m.session(80), m.session(80)
    a.eval(p)
    want, tokens = a.logits().copy(), a.generate(8)
    ctx.close()
    a.free()
    b.eval(p)
    assert np.array_equal(b.logits().view(np.uint32), want.view(np.uint32))
    assert np.array_equal(b.generate(8), tokens)
    c = m.session(80)                 # on a's memory
    c.eval(p)
    assert np.array_equal(c.logits().view(np.uint32), want.view(np.uint32))
    b.free()
    c.free()
    m.free()
