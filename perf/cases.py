"""The work that users of ornithology_amd have it do, as measurable cases.

Three groups, each through the public entry points of ``ornithology_amd``:

* the kernel-level calls on host buffers (``Tensor.matvec``,
  ``Context.quantize``), as the reference's matvec seam and GGUF tooling use them;
* requests: a session is opened on a loaded model, a prompt (and perhaps a
  second turn) is evaluated, tokens are generated, the logits are read, the
  session is closed;
* decode: one token step of an open session and its logits, as a program that
  samples on the host makes them.

The models are written as GGUF files with random blocks and loaded, once per
process, as a program keeps its weights: "tiny" is the all-Q8_0 test model,
"block" four layers of the 35B shape (three delta-net, one attention, 256
experts), "attn" one attention layer of that shape with a dense FFN, "iq2" one
delta-net layer of the 397B shape with IQ2_XXS experts. "whole" is the 35B
shape with all of its 40 layers, synthesised on the device. One-layer and
four-layer models have a 32768-token vocabulary, so that the layers and not the
head are what takes the time.
"""
import math
import os
import struct
import tempfile
from collections import OrderedDict
from pathlib import Path

import numpy as np
import torch

import ornithology_amd as oa

F32, Q8_0, Q4_K, Q6_K, IQ2_XXS = oa.F32, oa.Q8_0, oa.Q4_K, oa.Q6_K, oa.IQ2_XXS
TYPES = {"Q8_0": Q8_0, "Q4_K": Q4_K, "Q6_K": Q6_K, "IQ2_XXS": IQ2_XXS}

MODELS = {
    "tiny": dict(hidden=512, n_layers=4, vocab=4096, full_interval=4, nh=8, nkv=2, hd=64, nk=4, nv=8, dhead=64,
                 conv_k=4, ne=16, top_k=4, inter=256, t=Q8_0, t_v=Q8_0, t_down=Q8_0, t_exps=Q8_0),
    "block": dict(hidden=2048, n_layers=4, vocab=32768, full_interval=4, nh=16, nkv=2, hd=256, nk=16, nv=32, dhead=128,
                  conv_k=4, ne=256, top_k=8, inter=512, t=Q4_K, t_v=Q6_K, t_down=Q6_K, t_exps=Q4_K),
    "attn": dict(hidden=2048, n_layers=1, vocab=32768, full_interval=1, nh=16, nkv=2, hd=256, nk=16, nv=32, dhead=128,
                 conv_k=4, ne=0, top_k=0, inter=4096, t=Q4_K, t_v=Q6_K, t_down=Q6_K, t_exps=Q4_K),
    "iq2": dict(hidden=4096, n_layers=1, vocab=32768, full_interval=4, nh=32, nkv=2, hd=256, nk=16, nv=64, dhead=128,
                conv_k=4, ne=512, top_k=10, inter=1024, t=Q4_K, t_v=Q4_K, t_down=Q4_K, t_exps=IQ2_XXS),
    "whole": dict(hidden=2048, n_layers=40, vocab=248320, full_interval=4, nh=16, nkv=2, hd=256, nk=16, nv=32, dhead=128,
                  conv_k=4, ne=256, top_k=8, inter=512, t=Q4_K, t_v=Q6_K, t_down=Q6_K, t_exps=Q4_K),
}


def listed():
    return [
        # the smallest call: a whole tiny model, where launches and host work are the time
        {"name": "tiny request 32+64", "kind": "request", "model": "tiny", "prompt": 32, "turn": 0, "gen": 64},
        # the reference's matvec seam, at the head of the 35B shape, one column
        {"name": "matvec head q4k x1", "kind": "matvec", "type": "Q4_K", "cols": 2048, "rows": 248320, "columns": 1},
        # the same seam over a prompt's columns, an odd number of them
        {"name": "matvec q6k x333", "kind": "matvec", "type": "Q6_K", "cols": 2048, "rows": 4096, "columns": 333},
        # GGUF tooling: one projection encoded
        {"name": "encode q4k", "kind": "encode", "type": "Q4_K", "blocks": 16384},
        # the benchmark's decode step: 40 layers, head, 4096 positions of context
        {"name": "whole decode 4096", "kind": "decode", "model": "whole", "context": 4096},
        # the benchmark's prompt, as a request
        {"name": "whole prompt 4096", "kind": "request", "model": "whole", "prompt": 4096, "turn": 0, "gen": 0},
        # layers of the 35B shape: an ordinary prompt of odd length
        {"name": "block prompt 1003", "kind": "request", "model": "block", "prompt": 1003, "turn": 0, "gen": 0},
        # a short chat turn after a short prompt, and its first tokens
        {"name": "block request 61+37+8", "kind": "request", "model": "block", "prompt": 61, "turn": 37, "gen": 8},
        # decode at an ordinary context
        {"name": "block decode 700", "kind": "decode", "model": "block", "context": 700},
        # an attention layer in long-context decode
        {"name": "attn decode 32768", "kind": "decode", "model": "attn", "context": 32768},
        # a layer of the 397B shape (IQ2_XXS experts): a prompt and a decode step
        {"name": "iq2 prompt 500", "kind": "request", "model": "iq2", "prompt": 500, "turn": 0, "gen": 0},
        {"name": "iq2 decode 200", "kind": "decode", "model": "iq2", "context": 200},
    ]


def _log(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49)))))))


def draw(rng):
    kind = rng.choice(("matvec", "encode", "request", "request", "decode"))
    if kind == "matvec":
        t = rng.choice(("Q8_0", "Q4_K", "Q6_K", "IQ2_XXS"))
        columns = 1 if rng.random() < 0.5 else _log(rng, 2, 4 if t == "IQ2_XXS" else 512)
        cols = 256 * rng.choice((1, 2, 3, 4, 8, 11, 16, 32))
        return {"kind": kind, "type": t, "cols": cols, "rows": _log(rng, 1, 65536 if columns == 1 else 8192),
                "columns": columns}
    if kind == "encode":
        t = rng.choice(("Q8_0", "Q4_K", "Q6_K", "IQ2_XXS"))
        return {"kind": kind, "type": t, "blocks": _log(rng, 1, 4096 if t == "IQ2_XXS" else 16384)}
    if kind == "request":
        model = rng.choice(("tiny", "block", "attn", "iq2"))
        prompt = _log(rng, 1, 600 if model == "iq2" else 4096)
        return {"kind": kind, "model": model, "prompt": prompt,
                "turn": 0 if rng.random() < 0.6 else _log(rng, 1, 300), "gen": 0 if rng.random() < 0.5 else _log(rng, 1, 32)}
    model = rng.choice(("tiny", "block", "attn", "iq2"))
    return {"kind": kind, "model": model, "context": _log(rng, 1, {"attn": 32768, "iq2": 500}.get(model, 4096))}


# ---- weights ------------------------------------------------------------------------

def _tensors(c):
    """[(name, type, dims, low, high)] of a model: quantised projections (low
    and high None) and the F32 tensors, uniform over [low, high)."""
    H, V, qd, vd = c["hidden"], c["vocab"], c["nk"] * c["dhead"], c["nv"] * c["dhead"]
    cc, aq, kvd, I, ne, t = 2 * qd + vd, c["nh"] * c["hd"], c["nkv"] * c["hd"], c["inter"], c["ne"], c["t"]
    out = [("token_embd.weight", t, (H, V), None, None), ("output_norm.weight", F32, (H,), 0.9, 1.1),
           ("output.weight", t, (H, V), None, None)]
    for l in range(c["n_layers"]):
        b = f"blk.{l}."
        out += [(b + "attn_norm.weight", F32, (H,), 0.9, 1.1), (b + "post_attention_norm.weight", F32, (H,), 0.9, 1.1)]
        if l % c["full_interval"] == c["full_interval"] - 1:
            out += [(b + "attn_q.weight", t, (H, 2 * aq), None, None), (b + "attn_k.weight", t, (H, kvd), None, None),
                    (b + "attn_v.weight", c["t_v"], (H, kvd), None, None),
                    (b + "attn_q_norm.weight", F32, (c["hd"],), 0.9, 1.1),
                    (b + "attn_k_norm.weight", F32, (c["hd"],), 0.9, 1.1), (b + "attn_output.weight", t, (aq, H), None, None)]
        else:
            out += [(b + "attn_qkv.weight", t, (H, cc), None, None), (b + "ssm_conv1d.weight", F32, (c["conv_k"], cc), -0.2, 0.2),
                    (b + "ssm_a", F32, (c["nv"],), -0.8, -0.2), (b + "ssm_dt.bias", F32, (c["nv"],), -0.05, 0.05),
                    (b + "ssm_norm.weight", F32, (c["dhead"],), 0.9, 1.1), (b + "ssm_alpha.weight", t, (H, c["nv"]), None, None),
                    (b + "ssm_beta.weight", t, (H, c["nv"]), None, None), (b + "attn_gate.weight", t, (H, vd), None, None),
                    (b + "ssm_out.weight", t, (vd, H), None, None)]
        if not ne:
            out += [(b + "ffn_gate.weight", t, (H, I), None, None), (b + "ffn_up.weight", t, (H, I), None, None),
                    (b + "ffn_down.weight", c["t_down"], (I, H), None, None)]
            continue
        te, td = c["t_exps"], c["t_exps"] if c["t_exps"] == IQ2_XXS else c["t_down"]
        out += [(b + "ffn_gate_inp.weight", t, (H, ne), None, None), (b + "ffn_gate_exps.weight", te, (H, I, ne), None, None),
                (b + "ffn_up_exps.weight", te, (H, I, ne), None, None), (b + "ffn_down_exps.weight", td, (I, H, ne), None, None),
                (b + "ffn_gate_shexp.weight", t, (H, I), None, None), (b + "ffn_up_shexp.weight", t, (H, I), None, None),
                (b + "ffn_down_shexp.weight", c["t_down"], (I, H), None, None),
                (b + "ffn_gate_inp_shexp.weight", t, (H,), None, None)]
    return out


def _blocks(t, n, gen):
    """n weights as random GGUF blocks with a spread of about 0.02, on the GPU
    (bytes, one row per block): codes, scales and signs are uniform."""
    size, nb = {Q8_0: (34, 32), Q4_K: (144, 256), Q6_K: (210, 256), IQ2_XXS: (66, 256)}[t]
    w = torch.randint(0, 256, (n // nb, size), dtype=torch.uint8, generator=gen, device=gen.device)
    half = lambda v: torch.tensor(np.frombuffer(np.float16(v).tobytes(), np.uint8).copy(), device=gen.device)  # noqa: E731
    if t == Q8_0:
        w[:, :2] = half(2.7e-4)
    elif t == Q4_K:
        w[:, :2], w[:, 2:4] = half(7.75e-5), half(7.5 * 7.75e-5)
    elif t == Q6_K:
        w[:, 208:] = half(1.46e-5)
    else:
        w[:, :2] = half(5e-4)
    return w.reshape(-1)


def _gen(*key):
    g = torch.Generator(device="cuda" if torch.cuda.is_available() else "cpu")
    g.manual_seed(hash(key) & 0x7FFFFFFF)
    return g


def _data(name, k, t, dims, lo, hi):
    n = math.prod(dims)
    if lo is not None:
        return np.random.default_rng((list(MODELS).index(name), k)).uniform(lo, hi, n).astype(np.float32).view(np.uint8)
    return _blocks(t, n, _gen(list(MODELS).index(name), k))


def _write_gguf(path, name):
    """The random model `name` as a GGUF v3 file."""
    c = MODELS[name]
    text = lambda s: struct.pack("<Q", len(s)) + s.encode()  # noqa: E731
    u32 = lambda k, v: text(k) + struct.pack("<II", 4, v)  # noqa: E731
    f32 = lambda k, v: text(k) + struct.pack("<If", 6, v)  # noqa: E731
    a = "qwen35moe."
    kv = [text("general.architecture") + struct.pack("<I", 8) + text("qwen35moe"), u32(a + "block_count", c["n_layers"]),
          u32(a + "expert_used_count", c["top_k"]), u32(a + "rope.dimension_count", 64), f32(a + "rope.freq_base", 1e7),
          f32(a + "attention.layer_norm_rms_epsilon", 1e-6),
          text("tokenizer.ggml.tokens") + struct.pack("<IIQ", 9, 8, 0)]
    ts, off, head = _tensors(c), 0, b""
    for nm, t, dims, _, _ in ts:
        head += text(nm) + struct.pack("<I%dQIQ" % len(dims), len(dims), *dims, t, off)
        off += -(-oa.row_bytes(t, math.prod(dims)) // 32) * 32
    head = b"GGUF" + struct.pack("<IQQ", 3, len(ts), len(kv)) + b"".join(kv) + head
    with open(path, "wb") as f:
        f.write(head + b"\0" * (-len(head) % 32))
        for k, (_, t, dims, lo, hi) in enumerate(ts):
            d = _data(name, k, t, dims, lo, hi)
            d = d if isinstance(d, np.ndarray) else d.cpu().numpy()
            f.write(d.data)
            f.write(b"\0" * (-d.nbytes % 32))


class _Weights:
    """A model on the device, freed with its last user."""

    def __init__(self, name):
        c = MODELS[name]
        self.vocab = c["vocab"]
        if name == "whole":
            k = {x: c[x] for x in ("hidden", "n_layers", "vocab", "full_interval", "nh", "nkv", "hd", "nk", "nv", "dhead",
                                   "conv_k", "ne", "top_k")}
            self.model = _context().synth(**k, moe_inter=c["inter"], shared_inter=c["inter"], t_default=c["t"],
                                          t_attn_v=c["t_v"], t_ffn_down=c["t_down"], t_output=c["t"], t_embd=c["t"],
                                          seed=0, sigma=0.02)
        else:
            with tempfile.TemporaryDirectory() as d:
                _write_gguf(os.path.join(d, "model.gguf"), name)
                self.model = _context().load(os.path.join(d, "model.gguf"))
        self.model.session(64).free()   # what is laid out once per model is laid out here

    def __del__(self):
        try:
            self.model.free()
        except Exception:
            pass


class _Open:
    """An open session on a context of `context` tokens; opened again once it is full."""

    def __init__(self, weights, prompt, room):
        self.weights, self.prompt, self.room, self.s = weights, prompt, room, None

    def session(self, steps):
        if self.s is None or self.s.pos + steps > len(self.prompt) + self.room:
            self.close()
            self.s = self.weights.model.session(len(self.prompt) + self.room)
            self.s.eval(self.prompt)
        return self.s

    def close(self):
        if self.s is not None:
            self.s.free()
            self.s = None

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass


_ctx = None
_models = OrderedDict()   # the models in use, the oldest given up beyond five


def _context():
    global _ctx
    if _ctx is None:
        _ctx = oa.Context(0)
    return _ctx


def _weights(name):
    if name not in _models:
        while len(_models) >= 5:
            _models.popitem(last=False)
        _models[name] = _Weights(name)
    _models.move_to_end(name)
    return _models[name]


class _Tensor:
    def __init__(self, case, seed):
        t = TYPES[case["type"]]
        self.t = _context().upload("w", t, _blocks(t, case["cols"] * case["rows"], _gen(seed, 1)).cpu().numpy(),
                                   (case["cols"], case["rows"]))

    def __del__(self):
        try:
            self.t.free()
        except Exception:
            pass


def _tokens(case, seed):
    n = case.get("context", 0) + case.get("prompt", 0) + case.get("turn", 0) + 64
    return np.random.default_rng(seed).integers(0, MODELS[case["model"]]["vocab"], n).astype(np.int32)


# ---- the cases ------------------------------------------------------------------------

def prepare(case, seed):
    s = {"case": case}
    if case["kind"] == "matvec":
        s["w"] = _Tensor(case, seed)
        s["x"] = np.random.default_rng(seed).standard_normal(case["columns"] * case["cols"]).astype(np.float32)
    elif case["kind"] == "encode":
        s["ctx"] = _context()
        s["x"] = (0.02 * np.random.default_rng(seed).standard_normal(case["blocks"] * 256)).astype(np.float32)
    elif case["kind"] == "request":
        s["weights"], s["tokens"] = _weights(case["model"]), _tokens(case, seed)
    else:
        s["tokens"] = _tokens(case, seed)
        s["open"] = _Open(_weights(case["model"]), s["tokens"][:case["context"]], 1024 if case["model"] == "whole" else 4096)
        s["open"].session(1)
    return s


def run(state):
    c = state["case"]
    if c["kind"] == "matvec":
        return state["w"].t.matvec(state["x"])
    if c["kind"] == "encode":
        return state["ctx"].quantize(TYPES[c["type"]], state["x"])
    if c["kind"] == "request":
        p, t, g, tok = c["prompt"], c["turn"], c["gen"], state["tokens"]
        s = state["weights"].model.session(p + t + g)
        s.eval(tok[:p])
        if t:
            s.eval(tok[p:p + t])
        out = [s.logits()]
        if g:
            out += [s.generate(g), s.logits()]
        s.free()
        return out
    s = state["open"].session(1)
    s.step(int(state["tokens"][c["context"] + s.pos % 64]))
    return s.logits()


def work(case):
    if case["kind"] == "matvec":
        n, m, k = case["cols"], case["rows"], case["columns"]
        return {"bytes": oa.row_bytes(TYPES[case["type"]], n * m) + 4.0 * k * (n + m), "flops": 2.0 * n * m * k}
    if case["kind"] == "encode":
        n = 256 * case["blocks"]
        return {"bytes": 4.0 * n + oa.row_bytes(TYPES[case["type"]], n), "flops": 0.0}
    c = MODELS[case["model"]]
    start = case.get("context", 0)
    first, gen = (case["prompt"] + case["turn"], case["gen"]) if case["kind"] == "request" else (1, 0)
    cc, aq = 2 * c["nk"] * c["dhead"] + c["nv"] * c["dhead"], c["nh"] * c["hd"]
    total_b = total_f = 0.0
    for n, pos, heads in [(first, start, 1)] + [(1, start + first + k, 1) for k in range(gen)]:
        for nm, t, dims, lo, _ in _tensors(c):
            b, f = oa.row_bytes(t, math.prod(dims)), 0.0 if lo is not None else 2.0 * math.prod(dims)
            if nm.startswith("token_embd"):
                total_b += n * b / c["vocab"]
            elif nm.startswith("output"):
                total_b, total_f = total_b + b, total_f + f * heads
            elif "_exps" in nm:
                total_b += b * (1.0 - (1.0 - c["top_k"] / c["ne"]) ** n)   # experts that some token takes
                total_f += n * f * c["top_k"] / c["ne"]
            else:
                total_b, total_f = total_b + b, total_f + n * f
        for l in range(c["n_layers"]):
            if l % c["full_interval"] == c["full_interval"] - 1:
                total_b += 2 * (pos + n) * c["nkv"] * (c["hd"] + 4)
                total_f += 4.0 * aq * (n * pos + n * (n + 1) / 2)
            else:
                state = c["nv"] * c["dhead"] ** 2
                total_b += 8.0 * state + 8.0 * (c["conv_k"] - 1) * cc
                total_f += 6.0 * state * n
        total_b += 4.0 * c["vocab"]
    return {"bytes": total_b, "flops": total_f}


def tolerance(case):
    # Encoders give the reference's bytes.
    if case["kind"] == "encode":
        return "exact"
    # Integer products, float sums over the super-blocks of a row (or, IQ2_XXS,
    # over its elements): see exact(); about four times what is measured there.
    if case["kind"] == "matvec":
        return {"rel": 2e-6, "max": 2e-5}
    # Every layer rounds its activations to 8 bits per block. A last-bit difference
    # moves one code now and then, and that code moves others at the next rounding:
    # the logits of one layer and the head are then 0.014 to 0.019 from 64 bits (where
    # no code moves, 2e-7), those of four layers 0.005 to 0.031, and another order of
    # the sums (the matrix-core delta scan, flash attention) moves them by 0.005 to
    # 0.022. Greedy tokens are whole values.
    return {"rel": 0.03, "max": 0.3, "differ": 0.01}


# ---- the same in 64 bits -----------------------------------------------------------------

def _u16(b):
    return (b[..., 0].to(torch.int32) | (b[..., 1].to(torch.int32) << 8))


def _half(b):
    return b.contiguous().view(torch.float16).double().squeeze(-1)


def _dequant(t, w, n_in):
    """GGUF bytes -> [rows, n_in] in 64 bits."""
    if t == Q8_0:
        w = w.reshape(-1, 34)
        out = _half(w[:, :2])[:, None] * w[:, 2:].contiguous().view(torch.int8).double()
    elif t == Q4_K:
        w = w.reshape(-1, 144)
        s = w[:, 4:16].to(torch.int32)
        sc = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | ((s[:, :4] >> 6) << 4)], 1)
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1)
        q = w[:, 16:].reshape(-1, 4, 1, 32)
        q = torch.cat([q & 15, q >> 4], 2).reshape(-1, 8, 32).double()
        out = (_half(w[:, :2])[:, None] * sc)[..., None] * q - (_half(w[:, 2:4])[:, None] * mn)[..., None]
    elif t == Q6_K:
        w = w.reshape(-1, 210)
        ql, qh = w[:, :128].reshape(-1, 2, 2, 32).to(torch.int32), w[:, 128:192].reshape(-1, 2, 1, 32).to(torch.int32)
        q = torch.cat([(ql & 15) | (((qh >> torch.tensor([0, 2], device=w.device)[:, None]) & 3) << 4),
                       (ql >> 4) | (((qh >> torch.tensor([4, 6], device=w.device)[:, None]) & 3) << 4)], 2) - 32
        sc = w[:, 192:208].contiguous().view(torch.int8).double()
        out = (_half(w[:, 208:])[:, None] * sc)[..., None] * q.reshape(-1, 16, 16).double()
    else:
        text = (Path(oa.HERE).parent / "include" / "ornith_iq2xxs_grid.h").read_text()   # the codebook: data of the format
        grid = torch.tensor([[(int(v[:18], 16) >> (8 * j)) & 255 for j in range(8)] for v in text.split() if v.startswith("0x") and "ull" in v],
                            dtype=torch.float64, device=w.device)
        w = w.reshape(-1, 66)
        b = w[:, 2:].reshape(-1, 8, 8).to(torch.int64)
        a1 = b[..., 4] | (b[..., 5] << 8) | (b[..., 6] << 16) | (b[..., 7] << 24)
        sg = (a1[..., None] >> torch.tensor([0, 7, 14, 21], device=w.device)) & 127
        bits = (sg[..., None] >> torch.arange(7, device=w.device)) & 1
        bits = torch.cat([bits, bits.sum(-1, keepdim=True) & 1], -1)
        db = _half(w[:, :2])[:, None] * (0.5 + (a1 >> 28).double()) * 0.25
        out = db[..., None, None] * grid[b[..., :4]] * (1 - 2 * bits).double()
    return out.reshape(-1, n_in)


def _q8k(x):
    """Activations rounded to 8 bits per block of 256, as the integer products take them."""
    b = x.reshape(-1, 256)
    m = b.gather(1, b.abs().argmax(1, keepdim=True))
    s = torch.where(m == 0, torch.zeros_like(m), -127 / torch.where(m == 0, torch.ones_like(m), m))
    return torch.where(m == 0, torch.zeros_like(b), (b * s).round() / torch.where(s == 0, torch.ones_like(s), s)).reshape(x.shape)


def _mm(t, w, x):
    return (x if t == IQ2_XXS else _q8k(x)) @ _dequant(t, w, x.shape[-1]).T


def _norm(x, w):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + 1e-6) * w


def _layer64(c, W, l, x, last):
    """One layer over the tokens' rows x; only the last row where `last`."""
    P = lambda n: W[f"blk.{l}.{n}"]  # noqa: E731
    mm = lambda n, v: _mm(*P(n)[:2], v)  # noqa: E731
    f = lambda n: P(n)[1].view(torch.float32).double()  # noqa: E731
    T, hd, d = x.shape[0], c["hd"], c["dhead"]
    rows = slice(T - 1, T) if last else slice(0, T)
    xn = _norm(x, f("attn_norm.weight"))
    if l % c["full_interval"] == c["full_interval"] - 1:
        at = torch.arange(T, device=x.device, dtype=torch.float64)
        freq = (1e7 ** (-2.0 * torch.arange(32, device=x.device, dtype=torch.float64) / 64)).float()
        ang = (at.float()[:, None] * freq).double()   # angles are defined in 32 bits: a context's positions magnify theirs
        cos, sin = ang.cos()[:, None], ang.sin()[:, None]
        rope = lambda v, r: torch.cat([v[..., :32] * cos[r] - v[..., 32:64] * sin[r],  # noqa: E731
                                       v[..., :32] * sin[r] + v[..., 32:64] * cos[r], v[..., 64:]], -1)

        def q8(v):
            s = v.abs().amax(-1, keepdim=True) / 127
            return (v / s).round() * s

        qg = mm("attn_q.weight", xn[rows]).reshape(-1, c["nh"], 2, hd)
        q = rope(_norm(qg[:, :, 0], f("attn_q_norm.weight")), rows)
        k = q8(rope(_norm(mm("attn_k.weight", xn).reshape(T, c["nkv"], hd), f("attn_k_norm.weight")), slice(0, T)))
        v = q8(mm("attn_v.weight", xn).reshape(T, c["nkv"], hd))
        o = torch.empty_like(q)
        g = c["nh"] // c["nkv"]
        for h in range(c["nh"]):
            for r in range(0, q.shape[0], 2048):
                s = q[r:r + 2048, h] @ k[:, h // g].T / math.sqrt(hd)
                s = s.masked_fill(at[None, :] > at[rows][r:r + 2048, None], -math.inf)
                o[r:r + 2048, h] = s.softmax(-1) @ v[:, h // g]
        o = (o * qg[:, :, 1].sigmoid()).reshape(q.shape[0], -1)
        x = x[rows] + mm("attn_output.weight", o)
    else:
        qd, nv = c["nk"] * d, c["nv"]
        cat = mm("attn_qkv.weight", xn)
        w = f("ssm_conv1d.weight").reshape(-1, c["conv_k"])
        pad = torch.cat([cat.new_zeros(c["conv_k"] - 1, cat.shape[1]), cat])
        cv = sum(pad[j:j + T] * w[:, j] for j in range(c["conv_k"]))
        cv = cv * cv.sigmoid()
        l2 = lambda v: v * torch.rsqrt((v * v).sum(-1, keepdim=True) + 1e-6)  # noqa: E731
        heads = torch.arange(nv, device=x.device) % c["nk"]
        q, k = l2(cv[:, :qd].reshape(T, -1, d))[:, heads], l2(cv[:, qd:2 * qd].reshape(T, -1, d))[:, heads]
        v = cv[:, 2 * qd:].reshape(T, nv, d)
        al = torch.exp(f("ssm_a") * torch.nn.functional.softplus(mm("ssm_alpha.weight", xn) + f("ssm_dt.bias")))
        be = mm("ssm_beta.weight", xn).sigmoid()
        S, o = x.new_zeros(nv, d, d), torch.empty_like(v)
        for t in range(T):
            S = S * al[t, :, None, None]
            u = be[t, :, None] * (v[t] - (S @ k[t, :, :, None])[..., 0])
            S = S + u[:, :, None] * k[t, :, None, :]
            o[t] = (S @ q[t, :, :, None])[..., 0]
        z = mm("attn_gate.weight", xn[rows])
        o = _norm(o[rows] / math.sqrt(d), f("ssm_norm.weight")).reshape(z.shape) * (z * z.sigmoid())
        x = x[rows] + mm("ssm_out.weight", o)
    xn = _norm(x, f("post_attention_norm.weight"))
    act = lambda a, b: a * a.sigmoid() * b  # noqa: E731
    if not c["ne"]:
        return x + mm("ffn_down.weight", act(mm("ffn_gate.weight", xn), mm("ffn_up.weight", xn)))
    lg, pick = mm("ffn_gate_inp.weight", xn).topk(c["top_k"], -1)
    wt = lg.softmax(-1)
    y = mm("ffn_down_shexp.weight", act(mm("ffn_gate_shexp.weight", xn), mm("ffn_up_shexp.weight", xn)))
    y = y * mm("ffn_gate_inp_shexp.weight", xn).sigmoid()
    ex = lambda n, e: (P(n)[0], P(n)[1].reshape(c["ne"], -1)[e])  # noqa: E731
    for e in pick.unique().tolist():
        r, j = (pick == e).nonzero(as_tuple=True)
        h = act(_mm(*ex("ffn_gate_exps.weight", e), xn[r]), _mm(*ex("ffn_up_exps.weight", e), xn[r]))
        y.index_add_(0, r, wt[r, j][:, None] * _mm(*ex("ffn_down_exps.weight", e), h))
    return x + y


def exact(case, seed):
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    if case["kind"] == "encode" or case.get("model") == "whole":   # bytes; 40 layers take too long
        return None
    if case["kind"] == "matvec":
        t = TYPES[case["type"]]
        w = _blocks(t, case["cols"] * case["rows"], _gen(seed, 1)).to(dev)
        x = np.random.default_rng(seed).standard_normal(case["columns"] * case["cols"]).astype(np.float32)
        x = torch.from_numpy(x).to(dev).double().reshape(case["columns"], -1)
        rb, step = oa.row_bytes(t, case["cols"]), max(1, (1 << 27) // case["cols"])
        y = [_mm(t, w[r * rb:(r + step) * rb], x) for r in range(0, case["rows"], step)]
        return torch.cat(y, 1).reshape(-1).cpu().numpy()
    c, tok = MODELS[case["model"]], _tokens(case, seed)
    if case["kind"] == "request":
        tok = tok[:case["prompt"] + case["turn"]]
    else:
        n = case["context"]
        tok = np.append(tok[:n], tok[n + n % 64])
    W = {}
    for k, (nm, t, dims, lo, hi) in enumerate(_tensors(c)):
        d = _data(case["model"], k, t, dims, lo, hi)
        W[nm] = (t, torch.from_numpy(d).to(dev) if isinstance(d, np.ndarray) else d.to(dev))
    t, w = W["token_embd.weight"]
    x = _dequant(t, w.reshape(c["vocab"], -1)[torch.from_numpy(tok).long().to(dev)].reshape(-1), c["hidden"])
    for l in range(c["n_layers"]):
        x = _layer64(c, W, l, x, l == c["n_layers"] - 1)
    y = _mm(*W["output.weight"], _norm(x, W["output_norm.weight"][1].view(torch.float32).double()))[0].cpu().numpy()
    if case["kind"] == "decode":
        return y
    return [y, None, None] if case["gen"] else [y]   # tokens generated after a rounding are another text's
