"""What the speed of this framework is measured on: the RWKV-4-169M codec's own
calls, small to large, each through a public entry point.

The path has two directions. Compress runs packed windows (B streams x up to
1024 tokens: embed, 12 layers, head, softmax -> CDF interval, range coder);
decompress runs one token per stream per step with everything on the GPU. A
file is one to a few hundred chunks, so B goes from 1 (a small file, latency)
through tens (ragged last windows) to 256 and 512 (the benchmark's batch, the
engine's default). Both codecs (fp16, w8a8) are in use. Callers with a coder
of their own take logits (stepped or packed), CDF rows, or run single layers.

The model is the synthetic 169M shape (seed 0), loaded once as a program does;
tokens are Zipf(1.1) with 5% repeated spans, drawn from the case's seed.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from krunch_amd import _lib, cpp_path, krunch_ac_hip, synthetic
from krunch_amd.inference import InferenceEngine, coder_stream_cap
from krunch_amd.model import State

L, C, F, V = synthetic.N_LAYER, synthetic.N_EMBD, synthetic.N_FFN, synthetic.N_VOCAB
BOS, PRECISION = synthetic.BOS_TOKEN, 24
LAYER_WEIGHTS = 5 * C * C + 2 * C * F          # parameters of one layer's seven matrices
STATE_BYTES = 16 * C * L                       # recurrent state of one stream
DEV = "cuda"


def listed():
    return [
        # One stream scored or decoded token by token with the coder on the
        # host: graph-replayed single steps, the smallest call there is.
        {"name": "step_1", "kind": "step", "n": 16},
        # One layer op as the reference's extension is called, a mid-sized
        # [B, T, C] batch.
        {"name": "layer_8x128", "kind": "layer", "B": 8, "T": 128},
        # Full CDF rows for a caller's own coder; not a multiple of anything.
        {"name": "cdf_300", "kind": "cdf", "N": 300},
        # Packed logits of one text of 777 tokens (scoring, odd length).
        {"name": "packed_1x777", "kind": "packed", "B": 1, "T": 777},
        # A small file: one chunk, one window.
        {"name": "compress_1x1000", "kind": "compress", "q8": False, "B": 1, "T": 1000, "ragged": False},
        # A file of a few chunks of different lengths, two windows.
        {"name": "compress_20_ragged", "kind": "compress", "q8": False, "B": 20, "T": 1300, "ragged": True},
        # The int8 codec on a mid-sized file.
        {"name": "compress_q8_64x1024", "kind": "compress", "q8": True, "B": 64, "T": 1024, "ragged": False},
        # The benchmark's window: 256 chunks x 1024 tokens (the largest).
        {"name": "compress_256x1024", "kind": "compress", "q8": False, "B": 256, "T": 1024, "ragged": False},
        # Decompress of one chunk: latency of the step.
        {"name": "decode_1", "kind": "decode", "q8": False, "B": 1, "T": 64, "ragged": False},
        # Decompress of a few chunks of different lengths.
        {"name": "decode_40_ragged", "kind": "decode", "q8": False, "B": 40, "T": 64, "ragged": True},
        # The int8 codec's decompress.
        {"name": "decode_q8_128", "kind": "decode", "q8": True, "B": 128, "T": 64, "ragged": False},
        # The benchmark's decompress batch.
        {"name": "decode_256", "kind": "decode", "q8": False, "B": 256, "T": 64, "ragged": False},
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["step", "layer", "cdf", "packed", "compress", "compress", "compress",
                       "decode", "decode", "decode"])
    if kind == "step":
        return {"kind": kind, "n": rng.randint(4, 32)}
    if kind == "cdf":
        return {"kind": kind, "N": _log(rng, 1, 1024)}
    if kind in ("layer", "packed"):
        T = _log(rng, 1, 1500)
        return {"kind": kind, "B": _log(rng, 1, max(1, min(64, 4096 // T))), "T": T}
    q8, ragged = rng.random() < 0.35, rng.random() < 0.5
    if kind == "compress":
        T = _log(rng, 24, 1400)
        return {"kind": kind, "q8": q8, "B": _log(rng, 1, min(256, 200000 // T)), "T": T, "ragged": ragged}
    return {"kind": kind, "q8": q8, "B": _log(rng, 1, 512), "T": rng.randint(16, 64), "ragged": ragged}


# ------------------------------------------------------------------ inputs
_MODEL: dict = {}


def _weights():
    if "w" not in _MODEL:
        _MODEL["w"] = synthetic.make_weights()
    return _MODEL["w"]


def _engine(q8):
    if q8 not in _MODEL:
        _MODEL[q8] = InferenceEngine().load(_weights(), w8a8=q8)
    return _MODEL[q8]


def _lens(case, seed):
    B, T = case["B"], case["T"]
    if not case["ragged"]:
        return [T] * B
    rng = np.random.default_rng([seed, 7])
    lens = rng.integers(max(1, T // 4), T + 1, B)
    lens[int(rng.integers(B))] = T
    return [int(n) for n in lens]


def _streams(case, seed):
    toks = synthetic.zipf_tokens(case["B"], case["T"], seed_base=1000 * (seed + 1), repeat_rate=0.05)
    return [t[:n].copy() for t, n in zip(toks, _lens(case, seed))]


LAYER_MATS = (("Kw", C, C), ("Vw", C, C), ("Rw", C, C), ("Ow", C, C),
              ("fKw", C, F), ("fVw", F, C), ("fRw", C, C))


def _layer_inputs(case, seed):
    """x, state and weights of one layer on the CPU (fp16 and fp32 as the op takes them)."""
    g = torch.Generator().manual_seed(seed)
    B, T = case["B"], case["T"]
    rnd = lambda *s: torch.randn(*s, generator=g)
    uni = lambda *s: torch.rand(*s, generator=g)
    d = {"x": rnd(B, T, C).half(), "att_xx": rnd(B, C).half(), "aa": rnd(B, C), "bb": 0.5 + uni(B, C),
         "pp": rnd(B, C), "ffn_xx": rnd(B, C).half()}
    for ln in ("ln1", "ln2"):
        d[ln + "_w"], d[ln + "_b"] = (1 + 0.1 * rnd(C)).half(), (0.1 * rnd(C)).half()
    for tm in ("tm_k", "tm_v", "tm_r", "ftm_k", "ftm_r"):
        d[tm] = uni(C).half()
    d["decay"], d["first"] = -torch.exp(torch.linspace(-5.0, 3.0, C)), torch.full((C,), math.log(0.3))
    for name, k, n in LAYER_MATS:
        d[name] = (0.02 * rnd(k, n)).half()
    return d


LAYER_STATE = ("att_xx", "aa", "bb", "pp", "ffn_xx")
LAYER_ORDER = ("ln1_w", "ln1_b", "tm_k", "tm_v", "tm_r", "decay", "first", "Kw", "Vw", "Rw", "Ow",
               "ln2_w", "ln2_b", "ftm_k", "ftm_r", "fKw", "fVw", "fRw")


def _cdf_logits(case, seed):
    """Logits as a language model gives them: a normal body, some rows peaked."""
    g = torch.Generator().manual_seed(seed)
    N = case["N"]
    x = 2.0 * torch.randn(N, V, generator=g)
    peak = torch.randint(0, V, (N,), generator=g)
    x[torch.arange(N), peak] += 12.0 * torch.rand(N, generator=g)
    return x.half()


def prepare(case, seed):
    kind = case["kind"]
    if kind == "layer":
        return {"case": case, **{k: v.to(DEV) for k, v in _layer_inputs(case, seed).items()}}
    if kind == "cdf":
        return {"case": case, "logits": _cdf_logits(case, seed).to(DEV)}
    if kind == "compress":
        return {"case": case, "eng": _engine(case["q8"]), "streams": _streams(case, seed)}
    if kind in ("step", "packed"):
        W = _engine(False).weights
        B, T = case.get("B", 1), case.get("T", case.get("n"))
        toks = synthetic.zipf_tokens(B, T, seed_base=1000 * (seed + 1), repeat_rate=0.05)
        return {"case": case, "W": W, "tokens": toks, "ids": torch.from_numpy(toks).to(DEV),
                "state": cpp_path.fresh_state_batched(W, B)}
    # decode: the payloads, and the buffers a decoding program keeps
    eng, B, T = _engine(case["q8"]), case["B"], case["T"]
    P = eng.weights["prepared"]
    lens = _lens(case, seed)
    bits = [p[8:] for p in eng.compress_tokens_batched(_streams(case, seed))]
    offs = np.cumsum([0] + [len(b) for b in bits])
    i32 = dict(dtype=torch.int32, device=DEV)
    nbytes = _lib.lib().kr_decode_workspace_bytes(B, 1, C, F)
    return {"case": case, "P": P,
            "input": torch.from_numpy(np.frombuffer(b"".join(bits) + b"\0", dtype=np.uint8).copy()).to(DEV),
            "base": torch.from_numpy(offs[:-1].astype(np.int32)).to(DEV),
            "limits": torch.tensor([len(b) for b in bits], **i32),
            "n_tokens": torch.tensor(lens, **i32), "count": torch.zeros(B, **i32),
            "syms": torch.zeros(B, **i32), "tokens": torch.zeros((B, T), **i32),
            "ac": torch.zeros((B, 4), dtype=torch.uint32, device=DEV),
            "state": State(L, B, C, DEV), "x": torch.empty((B, C), dtype=torch.float16, device=DEV),
            "ws": torch.empty(nbytes, dtype=torch.uint8, device=DEV),
            "logits": torch.empty((B, cpp_path.logits_ld(V)), dtype=torch.float16, device=DEV)}


# --------------------------------------------------------------------- run
def _state_parts(st):
    """The recurrent state as a few tensors (views of its buffer)."""
    raw = st.buf.view(L, -1)
    n = st.B * C
    f = raw[:, 4 * n:].view(torch.float32).view(L, 3, st.B, C)
    return {"xx": raw[:, :4 * n].view(torch.float16).view(L, 2, st.B, C),
            "aa": f[:, 0], "bb": f[:, 1], "pp": f[:, 2]}


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "compress":
        payloads = s["eng"].compress_tokens_batched(s["streams"])
        out = np.zeros(case["B"] * (coder_stream_cap(case["T"]) + 8), dtype=np.uint8)
        data = b"".join(payloads)
        out[:len(data)] = np.frombuffer(data, dtype=np.uint8)
        return {"bytes": out, "lens": np.array([len(p) for p in payloads], dtype=np.int64)}
    if kind == "decode":
        return _run_decode(s)
    if kind == "cdf":
        return cpp_path.softmax_cdfs_per_row(s["logits"])
    if kind == "layer":
        out = krunch_ac_hip.rwkv4_layer_step_cpp(s["x"], *(s[k] for k in LAYER_STATE),
                                                 *(s[k] for k in LAYER_ORDER))
        return {"x": out, **{k: s[k] for k in LAYER_STATE}}
    s["state"].reset()
    if kind == "step":
        out = [cpp_path.forward_stepped_graphed(s["W"], int(t), s["state"]) for t in s["tokens"][0]]
        return {"logits": out, **_state_parts(s["state"])}
    logits = cpp_path.forward_packed_batched(s["W"], s["ids"], s["state"])
    return {"logits": logits, **_state_parts(s["state"])}


def _run_decode(s):
    B, T = s["case"]["B"], s["case"]["T"]
    st = _lib.stream_ptr()
    s["state"].reset()
    s["syms"].fill_(BOS)
    s["count"].zero_()
    n_in = s["input"].numel()
    _lib.call("kr_decode_init_batched", s["input"].data_ptr(), n_in, s["base"].data_ptr(),
              s["limits"].data_ptr(), s["ac"].data_ptr(), B, st)
    _lib.call("kr_decode_run", s["P"].ptr, B, s["state"].ptr, s["syms"].data_ptr(), s["x"].data_ptr(),
              s["ws"].data_ptr(), s["ws"].numel(), s["logits"].data_ptr(), s["logits"].shape[1],
              s["input"].data_ptr(), n_in, s["base"].data_ptr(), s["limits"].data_ptr(),
              s["ac"].data_ptr(), s["tokens"].data_ptr(), T, s["count"].data_ptr(),
              s["n_tokens"].data_ptr(), PRECISION, T, 1, 1, st)
    # the tokens, the last step's logits (without the row padding) and the state left behind
    return {"tokens": s["tokens"], "coder": s["ac"].view(torch.int32), "logits": s["logits"][:, :V],
            **_state_parts(s["state"])}


# -------------------------------------------------------------------- work
def work(case):
    """Weights are read once per window or step (a step's 261 MB do not stay
    on the chip until the next one), activations in and out once."""
    kind = case["kind"]
    layer_b = LAYER_WEIGHTS * (1 if case.get("q8") else 2)
    model_b = L * layer_b + 2 * C * V
    per_token = 2.0 * (L * LAYER_WEIGHTS + C * V)
    if kind == "cdf":
        return {"bytes": case["N"] * (2.0 * V + 4.0 * (V + 1)), "flops": 0.0}
    if kind == "layer":
        M = case["B"] * case["T"]
        return {"bytes": layer_b + M * C * 4.0 + case["B"] * C * 32.0, "flops": 2.0 * LAYER_WEIGHTS * M}
    if kind == "packed":
        M = case["B"] * case["T"]
        return {"bytes": model_b + M * 2.0 * (C + V) + case["B"] * 2.0 * STATE_BYTES, "flops": per_token * M}
    if kind == "step":
        return {"bytes": case["n"] * (model_b + 2.0 * (C + V) + 2.0 * STATE_BYTES), "flops": per_token * case["n"]}
    # a ragged batch's mean length is about 5/8 of the longest
    M = case["B"] * case["T"] * (0.625 if case["ragged"] else 1.0)
    if kind == "compress":
        windows = -(-case["T"] // 1024)
        return {"bytes": windows * model_b + M * (2.0 * C + 6.0), "flops": per_token * M}
    return {"bytes": case["T"] * model_b + M * (2.0 * STATE_BYTES + 2.0 * C + 4.0),
            "flops": per_token * M}


def tolerance(case):
    """Payloads, tokens, coder states and CDF rows are exact. Floating outputs
    round to fp16 between the stages of a layer: one layer is 3e-4 off its
    64-bit value, the 12-layer model 1.7e-3 (logits), and another order of the
    sums rounds as many values the other way; about four times that."""
    if case["kind"] in ("compress", "cdf"):
        return "exact"
    if case["kind"] == "layer":
        return {"rel": 1.5e-3}
    return {"rel": 8e-3}


# ------------------------------------------------------------------- exact
def _ln(x, w, b):
    m = x.mean(-1, keepdim=True)
    v = ((x - m) ** 2).mean(-1, keepdim=True)
    return (x - m) / torch.sqrt(v + 1e-5) * w + b


def _wkv64(k, v, w, u, aa, bb, pp):
    out = torch.empty_like(k)
    for t in range(k.shape[1]):
        kk, vv = k[:, t], v[:, t]
        ww = u + kk
        p = torch.maximum(pp, ww)
        e1, e2 = torch.exp(pp - p), torch.exp(ww - p)
        out[:, t] = (e1 * aa + e2 * vv) / (e1 * bb + e2)
        ww = w + pp
        p = torch.maximum(ww, kk)
        e1, e2 = torch.exp(ww - p), torch.exp(kk - p)
        aa, bb, pp = e1 * aa + e2 * vv, e1 * bb + e2, p
    return out, aa, bb, pp


def _layer64(x, att, aa, bb, pp, ffn, d):
    """One RWKV-4 layer over x [B, T, C] in float64; d holds its weights by the names above."""
    shift = lambda a, first: torch.cat([first.unsqueeze(1), a[:, :-1]], 1)
    mix = lambda a, s, tm: a * tm + s * (1 - tm)
    xx = _ln(x, d["ln1_w"], d["ln1_b"])
    sx = shift(xx, att)
    k, v = mix(xx, sx, d["tm_k"]) @ d["Kw"], mix(xx, sx, d["tm_v"]) @ d["Vw"]
    r = torch.sigmoid(mix(xx, sx, d["tm_r"]) @ d["Rw"])
    y, aa, bb, pp = _wkv64(k, v, d["decay"], d["first"], aa, bb, pp)
    att = xx[:, -1]
    x = x + (r * y) @ d["Ow"]
    xx = _ln(x, d["ln2_w"], d["ln2_b"])
    sx = shift(xx, ffn)
    kf = torch.relu(mix(xx, sx, d["ftm_k"]) @ d["fKw"]) ** 2
    x = x + torch.sigmoid(mix(xx, sx, d["ftm_r"]) @ d["fRw"]) * (kf @ d["fVw"])
    return x, att, aa, bb, pp, xx[:, -1]


def _forward64(ids, last_only):
    """The model from a fresh state in float64: logits and state parts as _state_parts lays them out."""
    w = _weights()
    up = lambda t: t.to(device=DEV, dtype=torch.float64)
    B = ids.shape[0]
    x = up(w["emb.weight"].to(DEV)[ids.to(DEV).long()])
    z = torch.zeros(B, C, dtype=torch.float64, device=DEV)
    xx, aas, bbs, pps = [], [], [], []
    for i in range(L):
        a, f, b = f"blocks.{i}.att.", f"blocks.{i}.ffn.", f"blocks.{i}."
        d = {"ln1_w": w[b + "ln1.weight"], "ln1_b": w[b + "ln1.bias"], "ln2_w": w[b + "ln2.weight"],
             "ln2_b": w[b + "ln2.bias"], "tm_k": w[a + "time_mix_k"], "tm_v": w[a + "time_mix_v"],
             "tm_r": w[a + "time_mix_r"], "ftm_k": w[f + "time_mix_k"], "ftm_r": w[f + "time_mix_r"],
             "decay": -torch.exp(w[a + "time_decay"].double()), "first": w[a + "time_first"],
             "Kw": w[a + "key.weight"], "Vw": w[a + "value.weight"], "Rw": w[a + "receptance.weight"],
             "Ow": w[a + "output.weight"], "fKw": w[f + "key.weight"], "fVw": w[f + "value.weight"],
             "fRw": w[f + "receptance.weight"]}
        x, att, aa, bb, pp, ffn = _layer64(x, z, z, z, z - 1e30, z, {k: up(t) for k, t in d.items()})
        xx.append(torch.stack([att, ffn]))
        aas.append(aa)
        bbs.append(bb)
        pps.append(pp)
    if last_only:
        x = x[:, -1:]
    logits = _ln(x, up(w["ln_out.weight"]), up(w["ln_out.bias"])) @ up(w["head.weight"])
    return logits, {"xx": torch.stack(xx), "aa": torch.stack(aas), "bb": torch.stack(bbs), "pp": torch.stack(pps)}


def exact(case, seed):
    kind = case["kind"]
    if kind in ("compress", "cdf") or case.get("q8"):
        return None                     # bytes and counts; quantised products have no plain 64-bit value
    if kind == "layer":
        d = {k: v.to(device=DEV, dtype=torch.float64) for k, v in _layer_inputs(case, seed).items()}
        out = _layer64(d["x"], d["att_xx"], d["aa"], d["bb"], d["pp"], d["ffn_xx"], d)
        return {"x": out[0], "att_xx": out[1], "aa": out[2], "bb": out[3], "pp": out[4], "ffn_xx": out[5]}
    if kind in ("step", "packed"):
        B, T = case.get("B", 1), case.get("T", case.get("n"))
        toks = synthetic.zipf_tokens(B, T, seed_base=1000 * (seed + 1), repeat_rate=0.05)
        logits, state = _forward64(torch.from_numpy(toks), False)
        return {"logits": list(logits[0]) if kind == "step" else logits.reshape(B * T, V), **state}
    # decode: inputs are BOS and the stream's own tokens; a finished stream repeats its last one
    B, T = case["B"], case["T"]
    ids = np.zeros((B, T), dtype=np.int64)
    for b, t in enumerate(_streams(case, seed)):
        ids[b, 1:len(t)] = t[:-1]
        ids[b, len(t):] = t[-1]
    logits, state = _forward64(torch.from_numpy(ids), True)
    return {"tokens": None, "coder": None, "logits": logits[:, 0], **state}
