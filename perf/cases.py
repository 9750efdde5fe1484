"""The calls that stand for what a user of the library has it do, at the sizes of BASELINE's configurations and of bench.py.

Kinds of case:
  op      the quantized-matrix operator on device tensors (pyre_qmatmul_dev), one matrix, 1..8 tokens
  moe     the MoE FFN block on device tensors (512 experts top-10 + shared), 1..8 tokens
  gdn     the Gated DeltaNet layer core over a prompt held in host arrays, recurrent state set before and read after it
  decode  greedy decoding of a few tokens behind a long context, then the logits a sampler would take over with
  verify  rounds of the speculative loop: a verify window's logits to the host, then the rollback to the kept tokens
  prompt  a prompt on an empty state, the last token's logits to the host
The last three run the A3B hybrid of the benchmark (48 layers, 512 experts) through the layer API.  Weights are random
blocks as everywhere in this repository; the model's are the same for every seed, as one loaded model serves every request.
"""
import math
import weakref

import numpy as np
import torch

from pyre_amd import lib, synth
from pyre_amd import modelgen as mg

TYPES = {"iq3_s": synth.IQ3_S, "iq2_xs": synth.IQ2_XS, "q4_k": synth.Q4_K, "q8_0": synth.Q8_0, "q6_k": synth.Q6_K, "q5_k": synth.Q5_K, "q3_k": synth.Q3_K,
         "iq4_xs": synth.IQ4_XS, "iq4_nl": synth.IQ4_NL, "iq3_xxs": synth.IQ3_XXS, "iq2_s": synth.IQ2_S, "iq2_xxs": synth.IQ2_XXS, "q4_0": synth.Q4_0, "q5_0": synth.Q5_0,
         "bf16": synth.BF16}
SWEEP = ("iq3_s", "iq2_xs", "q4_k", "q8_0")                      # the formats of the configurations' sweep
OTHER = tuple(t for t in TYPES if t not in SWEEP and t != "bf16")
MOST_CTX, MOST_PROMPT, MOST_OTHER = 32768, 8192, 512             # the last: prompts and contexts of models of other formats


def listed():
    return [
        # one projection for one token: the smallest call, where launches and latency count
        {"name": "op 4096x4096 iq3_s t1", "kind": "op", "type": "iq3_s", "rows": 4096, "cols": 4096, "t": 1},
        # the vocabulary head of one decode step (configs[1]; the GEMV bandwidth of the headline)
        {"name": "op head iq3_s t1", "kind": "op", "type": "iq3_s", "rows": 151936, "cols": 2048, "t": 1},
        # a drafter's head (the default draft vocabulary's rows: no whole number of tiles) for a verify window
        {"name": "op draft head q4_k t5", "kind": "op", "type": "q4_k", "rows": 40525, "cols": 2048, "t": 5},
        # the FFN block behind its own entry point
        {"name": "moe t4", "kind": "moe", "type": "iq3_s", "experts": 512, "d": 2048, "ff": 512, "t": 4},
        # a prompt through one Gated DeltaNet layer, with a remainder behind the last whole chunk
        {"name": "gdn prefill 4109", "kind": "gdn", "tokens": 4109},
        # chat: decoding behind a short and behind a long context (configs[4], the headline's loop)
        {"name": "decode ctx 900", "kind": "decode", "weights": "iq3_s", "mixes": "iq3_s", "ctx": 900, "tokens": 16},
        {"name": "decode ctx 32768", "kind": "decode", "weights": "iq3_s", "mixes": "iq3_s", "ctx": 32768, "tokens": 16},
        # the same model as files store it: hyper-connection matrices in bf16
        {"name": "decode bf16 mixes ctx 500", "kind": "decode", "weights": "iq3_s", "mixes": "bf16", "ctx": 500, "tokens": 16},
        # the speculative loop: four drafts a round, some of them kept
        {"name": "verify 5 ctx 4096", "kind": "verify", "weights": "iq3_s", "mixes": "iq3_s", "ctx": 4096, "width": 5, "rounds": 4},
        # a chat message and a document
        {"name": "prompt 301", "kind": "prompt", "weights": "iq3_s", "mixes": "iq3_s", "tokens": 301},
        {"name": "prompt 8192", "kind": "prompt", "weights": "iq3_s", "mixes": "iq3_s", "tokens": 8192},
        # a message for a model whose file is in another common format
        {"name": "prompt q4_k 200", "kind": "prompt", "weights": "q4_k", "mixes": "bf16", "tokens": 200},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choices(("op", "moe", "gdn", "decode", "verify", "prompt"), (6, 2, 1, 4, 3, 4))[0]
    if kind == "op":      # sizes of the sweep's shapes and everything between
        ty = rng.choice(SWEEP) if rng.random() < 0.7 else rng.choice(OTHER)
        return {"kind": kind, "type": ty, "rows": _log(rng, 512, 151936), "cols": 256 * _log(rng, 2, 16), "t": rng.randint(1, 8)}
    if kind == "moe":
        return {"kind": kind, "type": rng.choice(("iq3_s", "iq3_s", "iq3_s", "q4_k", "iq2_xs")), "experts": 32 * _log(rng, 2, 16), "d": 256 * _log(rng, 4, 8), "ff": 256 * rng.randint(1, 3), "t": rng.randint(1, 8)}
    if kind == "gdn":
        return {"kind": kind, "tokens": _log(rng, 16, 4109)}
    w, m = rng.choices((("iq3_s", "iq3_s"), ("iq3_s", "bf16"), ("q4_k", "bf16"), ("iq2_xs", "bf16")), (7, 2, 1, 1))[0]
    own = (w, m) == ("iq3_s", "iq3_s")
    c = {"kind": kind, "weights": w, "mixes": m}
    if kind == "prompt":
        return dict(c, tokens=_log(rng, 2, MOST_PROMPT if own else MOST_OTHER))
    c["ctx"] = _log(rng, 32, MOST_CTX if own else MOST_OTHER)
    if kind == "decode":
        return dict(c, tokens=rng.randint(8, 24))
    return dict(c, width=rng.randint(2, 8), rounds=rng.randint(2, 5))


# ---- what a program keeps: a context, and one model at a time -----------------------------------------------------------------
_ctx = None
_model = {"key": None, "model": None, "states": []}


def _context():
    global _ctx
    if _ctx is None:
        _ctx = lib.Context(0)
    return _ctx


def _cfg(case):
    return mg.a3b_config(qtype=TYPES[case["weights"]], hc_type=TYPES[case["mixes"]])


def _moe_cfg(case):
    return mg.a3b_config(qtype=TYPES[case["type"]], n_exp=case["experts"], d=case["d"], ff_exp=case["ff"])


def _bytes(ty, rows, cols):
    el, bs, _ = synth.GEOM[ty]
    return rows * (cols // el) * bs


def _the_model(case):
    """The model of the case's formats; the one of other formats goes first (two do not fit beside their loading)."""
    key = (case["weights"], case["mixes"])
    if _model["key"] == key:
        return _model["model"]
    for ref in _model["states"]:
        st = ref()
        if st is not None:
            st.close()
    if _model["model"] is not None:
        _model["model"].close()
    _model.update(key=None, model=None, states=[])
    ctx, c = _context(), _cfg(case)
    layers, globals_, raw = [dict() for _ in range(c.n_layers)], {}, []
    g = torch.Generator(device="cuda").manual_seed(3)
    for il, slot, kind, ty, rows, cols in mg.tensor_specs(c):
        if kind == "q" and ty == synth.BF16:
            w = torch.randn(rows, cols, device="cuda", generator=g).mul_(cols ** -0.5).bfloat16()
            raw.append(w)
            e = (ty, rows, cols, w.data_ptr())
        elif kind == "q":
            p = ctx.alloc(_bytes(ty, rows, cols))
            lo, hi = mg.scale_range(c, il, slot, ty)
            ctx.synth_blocks(ty, rows * (cols // synth.GEOM[ty][0]), mg.tensor_seed(1, il, slot), lo, hi, dev_out=p)
            raw.append(p)
            e = (ty, rows, cols, p)
        else:
            e = (ty, rows, cols, mg.host_tensor(c, 1, il, slot, kind, ty, rows, cols))
        (layers[il] if il >= 0 else globals_)[slot] = e
    torch.cuda.synchronize()
    m = lib.Model(ctx, c, layers, globals_)
    ctx.sync()
    for p in raw:
        if isinstance(p, int):
            ctx.free(p)
    del raw, layers, globals_
    torch.cuda.empty_cache()
    _model.update(key=key, model=m)
    return m


def _new_state(m, cap):
    st = m.new_state(cap)
    _model["states"] = [r for r in _model["states"] if r() is not None] + [weakref.ref(st)]
    return st


def _qmat(ty, rows, cols, seed):
    ctx = _context()
    n = _bytes(ty, rows, cols)
    b = torch.empty(n, dtype=torch.uint8, device="cuda")
    torch.cuda.synchronize()
    div = mg.WIDE_TYPES.get(ty, 1.0)
    ctx.synth_blocks(ty, rows * (cols // synth.GEOM[ty][0]), seed, 1e-3 / div, 2e-2 / div, dev_out=b.data_ptr())
    q = lib.QMat(ctx, ty, rows, cols, dev_blocks=b.data_ptr(), nbytes=n)
    ctx.sync()
    return q


def _normal(shape, seed, std=1.0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn(shape, device="cuda", generator=g).mul_(std)


def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case, "kind": kind}
    if kind == "op":
        s["m"] = _qmat(TYPES[case["type"]], case["rows"], case["cols"], 7000 + seed)
        s["x"] = _normal((case["t"], case["cols"]), seed)
        s["y"] = torch.empty(case["t"], case["rows"], device="cuda")
    elif kind == "moe":
        c = _moe_cfg(case)
        q = lambda rows, cols, k: _qmat(c.qtype, rows, cols, 16 * seed + k)
        router = _normal((c.n_exp, c.d), seed + 1, 0.02).bfloat16().cpu().view(torch.uint8).numpy().reshape(-1)
        s["m"] = lib.Moe(_context(), c.top_k, lib.QMat(_context(), synth.BF16, c.n_exp, c.d, router), q(c.n_exp * c.ff_exp, c.d, 0), q(c.n_exp * c.ff_exp, c.d, 1),
                         q(c.n_exp * c.d, c.ff_exp, 2), _normal((c.d,), seed + 2, 0.02).cpu().numpy(), q(c.ff_exp, c.d, 3), q(c.ff_exp, c.d, 4), q(c.d, c.ff_exp, 5))
        s["x"] = _normal((case["t"], c.d), seed)
        s["y"] = torch.empty(case["t"], c.d, device="cuda")
    elif kind == "gdn":
        nk, nv, t = 16, 32, case["tokens"]
        ch = 2 * nk * 128 + nv * 128
        host = lambda shape, k, std=1.0: _normal(shape, 8 * seed + k, std).cpu().numpy()
        g = np.random.Generator(np.random.PCG64(seed))
        a = -np.exp(g.uniform(0.0, np.log(16.0), nv))
        s["g"] = lib.Gdn(_context(), nk, nv, 128, 128, 4, 1e-6, a, np.zeros(nv), host((ch * 4,), 0, 0.5), 1 + host((128,), 1, 0.1))
        s["s0"] = host((nv, 128, 128), 2, 0.01)
        s["in"] = [host((t, ch), 3), host((t, nv * 128), 4), host((t, nv), 5), host((t, nv), 6)]
    else:
        m = _the_model(case)
        g = np.random.Generator(np.random.PCG64(seed))
        s["m"] = m
        ids = lambda n: g.integers(0, m.vocab, n, dtype=np.uint32)
        if kind == "prompt":
            s["ids"] = ids(case["tokens"])
            s["st"] = _new_state(m, case["tokens"])
        else:
            s["st"] = st = _new_state(m, case["ctx"] + 64)
            s["logits"] = m.forward(ids(case["ctx"]), st)
            s["snap"] = st.snapshot()
            if kind == "verify":
                s["windows"] = [ids(case["width"]) for _ in range(case["rounds"])]
                s["keep"] = [1 + int(g.integers(0, case["width"])) for _ in range(case["rounds"])]
    torch.cuda.synchronize()
    return s


def run(s):
    kind = s["kind"]
    if kind == "op":
        s["m"].matmul_dev(s["x"], s["case"]["t"], s["y"])
        return s["y"]
    if kind == "moe":
        s["m"].ffn_dev(s["x"], s["case"]["t"], s["y"])
        return s["y"]
    if kind == "gdn":
        s["g"].set_state(None, s["s0"])
        out = s["g"].prefill_chunked(*s["in"])
        return (out,) + s["g"].get_state()
    m, st = s["m"], s["st"]
    if kind == "prompt":
        st.reset()
        return m.forward(s["ids"], st)
    st.restore(s["snap"])                     # a request that goes on from a kept prompt
    if kind == "decode":
        toks, _ = m.generate_greedy(st, s["logits"], s["case"]["tokens"])
        return toks.astype(np.int64), m.forward(toks[-1:], st)
    outs = []
    for ids, keep in zip(s["windows"], s["keep"]):
        outs.append(m.forward_multi(ids, st))
        m.spec_keep(st, ids.size, keep)
    return outs


# ---- what a pass cannot do without --------------------------------------------------------------------------------------------
def _model_work(c, t, pos, logits):
    """(bytes, flops) of t tokens in one pass over the weights behind `pos` cached positions, `logits` rows of the head."""
    b, f = 0.0, 0.0
    for il, slot, kind, ty, rows, cols in mg.tensor_specs(c):
        n = _bytes(ty, rows, cols)
        if slot in (mg.GATE_E, mg.UP_E, mg.DOWN_E) and il >= 0:      # expected number of distinct experts of t tokens
            b += n * (1.0 - (1.0 - c.top_k / c.n_exp) ** t)
            f += 2.0 * rows * cols * c.top_k / c.n_exp * t
        elif il < 0 and slot == mg.G_EMBD:
            b += n / rows * t
        else:
            b += n
            f += 2.0 * rows * cols * (logits if il < 0 and slot == mg.G_OUT else t) * (kind in ("q", "router"))
    row, n_attn = c.n_kv * c.hd, c.n_layers // c.full_every
    n_lin = c.n_layers - n_attn
    old = max(0, pos - c.kv_recent) // 64 * 64
    b += n_attn * 2 * row * (0.625 * old + 4 * (pos - old) + 4 * t) + n_lin * 2 * (c.lin_nv * c.lin_dk * c.lin_dv + (c.conv_k - 1) * c.ch) * 4 + 4.0 * logits * c.vocab
    f += n_attn * 4.0 * c.n_head * c.hd * t * (pos + (t + 1) / 2) + n_lin * 8.0 * c.lin_nv * c.lin_dk * c.lin_dv * t
    return b, f


def work(case):
    kind = case["kind"]
    if kind == "op":
        r, c, t = case["rows"], case["cols"], case["t"]
        return {"bytes": _bytes(TYPES[case["type"]], r, c) + 4 * t * (r + c), "flops": 2 * r * c * t}
    if kind == "moe":
        c, t = _moe_cfg(case), case["t"]
        one = 2 * _bytes(c.qtype, c.ff_exp, c.d) + _bytes(c.qtype, c.d, c.ff_exp)
        return {"bytes": c.n_exp * c.d * 2 + one * (1 + c.n_exp * (1 - (1 - c.top_k / c.n_exp) ** t)) + 8 * t * c.d, "flops": t * (2 * c.n_exp * c.d + 6 * (c.top_k + 1) * c.d * c.ff_exp)}
    if kind == "gdn":
        t, nv, ch = case["tokens"], 32, 8192
        return {"bytes": 4 * (t * (ch + 2 * nv * 128 + 2 * nv) + 2 * nv * 128 * 128 + 2 * 3 * ch), "flops": t * (8 * nv * 128 * 128 + 8 * ch)}
    c = _cfg(case)
    if kind == "prompt":
        parts = [_model_work(c, case["tokens"], 0, 1)]
    elif kind == "decode":
        parts = [_model_work(c, 1, case["ctx"] + i, 1) for i in (0, case["tokens"] - 1)] * ((case["tokens"] + 1) // 2)
        parts = parts[:case["tokens"]]
    else:
        parts = [_model_work(c, case["width"], case["ctx"], case["width"])] * case["rounds"]
    return {"bytes": sum(p[0] for p in parts), "flops": sum(p[1] for p in parts)}


def tolerance(case):
    """Operators and blocks: f32 sums over a few thousand terms (activations and integer forms carry 22 bits).  The model:
    such differences pass 48 layers of normalisations, a 4-bit cache whose roundings they can tip, and a router whose
    last choice they can tip; its logits are held to the 1e-3 the model's parity is stated in, its tokens are whole."""
    kind = case["kind"]
    if kind == "op":
        return {"rel": 1e-5}
    if kind in ("moe", "gdn"):
        return {"rel": 2e-5, "max": 2e-3}
    return {"rel": 1e-3, "max": 2e-2, "differ": 0.0}
