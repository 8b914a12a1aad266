"""GPU: a prompt's IQ2_XXS experts grouped by expert (oh_kernels_iq2.hip) where
its branches part and beside other types:

* the rows kernel itself over given lists, against the oracle's rows: rows that
  do not fill a block of 256, pieces of every size of groups of 4 and of 8,
  with and without silu(gate) * up;
* models whose gate and up projections are IQ2_XXS and whose down projections
  are not, and the reverse;
* the sizes where the rule starts to group small experts that get few slots;
* tokens that pick one expert twice (a router with NaN logits).

Bar: the same bits as the oracle's rows, or as the token-by-token path."""
import ctypes as C

import numpy as np
import pytest

import clibs
import ornithology_amd as oa
from test_gpu_prefill import IQ2X, MIX, same_state, u32

pytestmark = pytest.mark.gpu


class Rows(C.Structure):              # oh_iq2rows (oh_types.h)
    _fields_ = [(n, C.c_void_p) for n in ("A", "C", "A2", "C2", "x", "y", "off", "list", "items")] + [
        (n, C.c_int) for n in ("n_in", "rows", "xstride", "ystride", "adiv", "cols")]


class Device:
    def __init__(self):
        self.ps = []

    def put(self, a):
        L, p, a = oa.lib(), C.c_void_p(), np.ascontiguousarray(a)
        assert L.hipMalloc(C.byref(p), C.c_size_t(a.nbytes)) == 0
        self.ps.append(p)
        assert L.hipMemcpy(p, C.c_void_p(a.ctypes.data), C.c_size_t(a.nbytes), 1) == 0
        return p

    def get(self, p, like):
        out = np.empty_like(like)
        assert oa.lib().hipMemcpy(C.c_void_p(out.ctypes.data), p, C.c_size_t(out.nbytes), 2) == 0
        return out

    def free(self):
        for p in self.ps:
            oa.lib().hipFree(p)


@pytest.mark.parametrize("pair", [False, True], ids=["rows", "pair"])
@pytest.mark.parametrize("rows,n_in,cols", [(1, 256, 8), (255, 512, 4), (257, 768, 8), (300, 256, 8), (512, 256, 4)])
def test_rows_match_oracle(hip_ctx, orc, rows, n_in, cols, pair):
    ne, adiv = 6, 3
    # experts of 0, 1, 2, 3, 4 and 13 slots, in mixed order
    idx = np.random.default_rng(rows).permutation(np.repeat(np.arange(ne), (0, 1, 2, 3, 4, 13))).astype(np.int32)
    idx = np.append(idx, np.int32(5))
    n = idx.size
    w = []
    for k in range(2 if pair else 1):
        b = np.random.default_rng(n_in + k).integers(0, 256, (ne * rows * n_in // 256, 66), np.uint8)
        b[:, :2] = np.frombuffer(np.float16(5e-4).tobytes(), np.uint8)
        w.append(b)
    x = clibs.gauss(4, f"x.{n_in}", n // adiv * n_in).reshape(-1, n_in)
    want = np.zeros((n, rows), np.float32)
    for p, e in enumerate(idx):
        ys = []
        for wk in w:
            y = np.zeros(rows, np.float32)
            we = np.ascontiguousarray(wk.reshape(ne, -1)[e])
            orc.orc_matvec(clibs.IQ2_XXS, clibs.bp(we), n_in, rows, clibs.f32p(np.ascontiguousarray(x[p // adiv])),
                           clibs.f32p(y), 0, 1)
            ys.append(y)
        want[p] = [np.float32(orc.orc_silu(float(g))) * u for g, u in zip(*ys)] if pair else ys[0]
    d, L = Device(), oa.lib()
    i32 = lambda m: d.put(np.zeros(m, np.int32))  # noqa: E731
    items = n // cols + min(ne, n)
    off, lst, its, err = i32(ne + 1), i32(n), i32(1 + items), i32(1)
    assert L.oh_launch_slot_lists(d.put(idx), n, ne, cols, off, lst, its, err, None) == 0
    planes = [d.put(b) for wk in w for b in (wk[:, 2:], wk[:, :2])] + [None, None]
    y = d.put(np.full((n, rows), np.nan, np.float32))
    r = Rows(*planes[:4], d.put(x), y, off, lst, its, n_in, rows, n_in, rows, adiv, cols)
    assert L.oh_launch_iq2_slots(C.byref(r), items, None) == 0
    hip_ctx.sync()
    got = d.get(y, want)
    d.free()
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))


class Mixed:
    """Two device models' tensors: `names` of the second, the rest of the first."""

    def __init__(self, a, b, names):
        self.pick = lambda n: b if n.endswith(names) else a

    def tensor_info(self, n):
        return self.pick(n).tensor_info(n)

    def tensor(self, n):
        return self.pick(n).tensor(n)


def both_paths(m, prompt, monkeypatch):
    out = []
    for prefill in ("1", "0"):
        monkeypatch.setenv("ORNITH_HIP_PREFILL", prefill)
        s = m.session(prompt.size + 8)
        s.eval(prompt)
        out.append(s)
    return out


@pytest.mark.parametrize("iq2", ["gate-up", "down", "up"])
def test_mixed_expert_types_equal_token_path(hip_ctx, tmp_path, monkeypatch, iq2):
    """300 tokens, top 2 of 8: 600 slots, past the 480 where they are grouped."""
    cfg = dict(MIX, n_layers=2, full_interval=2, seed=21)
    names = {"gate-up": ("ffn_gate_exps.weight", "ffn_up_exps.weight"), "down": ("ffn_down_exps.weight",),
             "up": ("ffn_up_exps.weight", "ffn_down_exps.weight")}[iq2]
    a, b = hip_ctx.synth(**cfg), hip_ctx.synth(**dict(cfg, t_exps=clibs.IQ2_XXS))
    path = tmp_path / "m.gguf"
    clibs.write_model_gguf(Mixed(a, b, names), cfg, path)
    a.free()
    b.free()
    m = hip_ctx.load(path)
    for t, n in zip(("gate", "up", "down"), ("ffn_gate_exps.weight", "ffn_up_exps.weight", "ffn_down_exps.weight")):
        assert (m.tensor_info("blk.0." + n)["type"] == clibs.IQ2_XXS) == (n in names), t
    sp, st = both_paths(m, np.random.default_rng(1).integers(0, cfg["vocab"], 300).astype(np.int32), monkeypatch)
    assert np.array_equal(u32(sp.logits()), u32(st.logits()))
    same_state(m, sp, st)
    sp.free()
    st.free()
    m.free()


@pytest.fixture(scope="module")
def thin(hip_ctx):
    m = hip_ctx.synth(**dict(IQ2X, n_layers=1, full_interval=2, ne=1024, top_k=8, moe_inter=256, shared_inter=256, seed=23))
    yield m
    m.free()


@pytest.mark.parametrize("n", [59, 94, 95, 226])
def test_small_thin_experts_equal_token_path(thin, monkeypatch, n):
    """1024 experts of 768 -> 256, top 8: 472 and 752 slots keep the rows, 760
    and 1808 (4 at a time: 1.8 slots an expert) are grouped."""
    sp, st = both_paths(thin, np.random.default_rng(n).integers(0, thin.arch["vocab"], n).astype(np.int32), monkeypatch)
    assert np.array_equal(u32(sp.logits()), u32(st.logits()))
    same_state(thin, sp, st)
    sp.free()
    st.free()


@pytest.mark.parametrize("ne", [8, 256])
def test_repeated_picks_equal_token_path(hip_ctx, tmp_path, monkeypatch, ne):
    """A router that gives NaN for every expert but the first: each of 300
    tokens picks expert 0 twice (once as the fallback, with weight 0), 600 slots
    of one expert."""
    cfg = dict(IQ2X, n_layers=2, full_interval=2, ne=ne, moe_inter=256, shared_inter=256, seed=25)
    a = hip_ctx.synth(**cfg)
    path = tmp_path / "m.gguf"
    clibs.write_model_gguf(a, cfg, path)
    a.free()
    raw = path.read_bytes()
    for l in range(cfg["n_layers"]):
        router = clibs.gguf_tensors(path)[f"blk.{l}.ffn_gate_inp.weight"][2]
        at = raw.index(router.tobytes())
        rows = router.reshape(ne, -1, 144)
        rows[1:, :, :2] = (0x00, 0x7E)                       # the scale d of Q4_K blocks: NaN
        raw = raw[:at] + rows.tobytes() + raw[at + router.nbytes:]
    path.write_bytes(raw)
    m = hip_ctx.load(path)
    sp, st = both_paths(m, np.random.default_rng(2).integers(0, cfg["vocab"], 300).astype(np.int32), monkeypatch)
    assert np.isfinite(sp.logits()).all() and sp.logits().any()
    assert np.array_equal(u32(sp.logits()), u32(st.logits()))
    same_state(m, sp, st)
    sp.free()
    st.free()
    m.free()
