"""GPU: the lists of (token, expert) slots by expert (oh_launch_slot_lists) that
the grouped IQ2_XXS experts of a prompt run over, against the same lists formed
on the host: duplicate picks, experts without slots, counts around whole
pieces. An index outside [0, ne) is left out and reported, and nothing is
written outside the lists."""
import ctypes as C

import numpy as np
import pytest

import ornithology_amd as oa

pytestmark = pytest.mark.gpu

EXPERT_LIST = 2                       # OH_ERR_EXPERT_LIST (oh_types.h)
GUARD, MARK = 64, -7


class Ints:
    """n device int32 with GUARD marked ones on both sides."""

    def __init__(self, n, data=None):
        self.n, self.p = n, C.c_void_p()
        host = np.full(n + 2 * GUARD, MARK, np.int32)
        if data is not None:
            host[GUARD:GUARD + n] = data
        L = oa.lib()
        assert L.hipMalloc(C.byref(self.p), C.c_size_t(host.nbytes)) == 0
        assert L.hipMemcpy(self.p, C.c_void_p(host.ctypes.data), C.c_size_t(host.nbytes), 1) == 0

    @property
    def at(self):
        return C.c_void_p(self.p.value + 4 * GUARD)

    def read(self):
        host = np.zeros(self.n + 2 * GUARD, np.int32)
        L = oa.lib()
        assert L.hipMemcpy(C.c_void_p(host.ctypes.data), self.p, C.c_size_t(host.nbytes), 2) == 0
        assert (host[:GUARD] == MARK).all() and (host[GUARD + self.n:] == MARK).all()
        L.hipFree(self.p)
        return host[GUARD:GUARD + self.n]


@pytest.mark.parametrize("bad", [(), (-1,), (0x7FFFFFFF, -0x80000000, "ne", 1023, 1024, 4096)],
                         ids=["valid", "one-bad", "bad"])
@pytest.mark.parametrize("ne,n,cols", [(8, 480, 4), (8, 1803, 8), (512, 2000, 8), (1024, 5000, 4)])
def test_slot_lists(hip_ctx, ne, n, cols, bad):
    rng = np.random.default_rng(ne + n)
    idx = np.minimum(rng.integers(0, ne, n), rng.integers(0, ne, n)).astype(np.int32)   # uneven
    idx[:cols + 1] = 0
    idx[-1] = ne - 1
    bad = [ne if b == "ne" else b for b in bad]
    bad = [b for b in bad if not 0 <= b < ne]
    for k, b in enumerate(bad):
        idx[20 + 37 * k] = b
    items_max = n // cols + min(ne, n)
    d = Ints(n, idx), Ints(ne + 1), Ints(n), Ints(1 + items_max), Ints(1, [0])
    L = oa.lib()
    assert L.oh_launch_slot_lists(d[0].at, n, ne, cols, d[1].at, d[2].at, d[3].at, d[4].at, None) == 0
    hip_ctx.sync()
    _, off, lst, items, err = [x.read() for x in d]
    assert err[0] == (EXPERT_LIST if bad else 0)
    good = (idx >= 0) & (idx < ne)
    counts = np.bincount(idx[good], minlength=ne)
    assert np.array_equal(off, np.concatenate([[0], np.cumsum(counts)]))
    for e in range(ne):
        assert np.array_equal(np.sort(lst[off[e]:off[e + 1]]), np.flatnonzero(good & (idx == e)))
    pieces = [(k << 10) | e for e in range(ne) for k in range(-(-int(counts[e]) // cols))]
    assert items[0] == len(pieces) and sorted(items[1:1 + items[0]]) == sorted(pieces)
