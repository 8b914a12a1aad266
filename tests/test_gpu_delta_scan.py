"""GPU: the prompt's chunked delta scan in the reference's order
(oh_k_delta_coef + oh_k_delta_chunked, src/ornith_attn.c:215-349) where its
branches part: prompts of one token, one short of a chunk, a chunk, one more,
and several chunks with a partial last one; and layers whose keys or values are
exactly zero for some heads or rows, which take the forms that skip zero terms
(the reference skips a term whose factor is zero, which matters for the sign of
a zero). Bar: logits and delta state bit-identical to the oracle's chunked
mode."""
import ctypes as C

import numpy as np
import pytest

import clibs
from clibs import i32p

pytestmark = pytest.mark.gpu

DK128 = dict(clibs.C1, hidden=768, n_layers=2, full_interval=2, vocab=1000, nh=4, nkv=1, hd=128, nk=2, nv=4, dhead=128,
             ne=8, top_k=2, moe_inter=512, shared_inter=512, t_default=clibs.Q4_K, t_attn_v=clibs.Q6_K,
             t_ffn_down=clibs.Q6_K, t_output=clibs.Q6_K, t_embd=clibs.Q4_K, seed=5)
DK64 = dict(clibs.C1, n_layers=2, full_interval=2)


def zero_rows(path, cfg):
    """Zero rows of the file's layer 0 attn_qkv: key head 0's keys, all values
    of value head 1, every third value row of value head 2."""
    data = clibs.gguf_tensors(path)["blk.0.attn_qkv.weight"][2]
    raw = path.read_bytes()
    at = raw.index(data.tobytes())
    d, nk = cfg["dhead"], cfg["nk"]
    rows = data.reshape(2 * nk * d + cfg["nv"] * d, -1)
    rows[nk * d:nk * d + d] = 0
    v = rows[2 * nk * d:]
    v[d:2 * d] = 0
    v[2 * d:3 * d:3] = 0
    path.write_bytes(raw[:at] + rows.tobytes() + raw[at + data.nbytes:])


@pytest.mark.parametrize("zeros", [False, True], ids=["plain", "zeros"])
@pytest.mark.parametrize("cfg", [DK64, DK128], ids=["dk64", "dk128"])
def test_chunked_scan_matches_oracle(hip_ctx, orc, tmp_path, monkeypatch, cfg, zeros):
    monkeypatch.setenv("ORNITH_PREFILL_SERIAL", "0")
    path = tmp_path / "m.gguf"
    clibs.write_c1_gguf(path, cfg)
    if zeros:
        zero_rows(path, cfg)
    om = C.c_void_p()
    assert orc.orc_model_load(str(path).encode(), C.byref(om)) == 0
    orc.orc_model_set_threads(om, 8)
    m = hip_ctx.load(path)
    rng = np.random.default_rng(2)
    for n in (1, 31, 32, 33, 141):
        p = rng.integers(0, cfg["vocab"], n).astype(np.int32)
        os_ = orc.orc_session_new(om, n, 1)
        assert orc.orc_session_eval(os_, i32p(p), n, 0) == 0
        s = m.session(n)
        s.eval(p)
        want = np.ctypeslib.as_array(orc.orc_session_logits(os_), (cfg["vocab"],))
        state = np.ctypeslib.as_array(orc.orc_session_delta(os_, 0), (cfg["nv"] * cfg["dhead"] ** 2,))
        assert np.array_equal(s.delta_state(0).view(np.uint32), state.view(np.uint32)), n
        assert np.array_equal(s.logits().view(np.uint32), want.view(np.uint32)), n
        s.free()
        orc.orc_session_free(os_)
    m.free()
    orc.orc_model_free(om)
