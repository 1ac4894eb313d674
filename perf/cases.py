"""Performance cases of the block-floating-point decode datapath.

Each case is one piece of work that a program using this package has it do,
through the public entry points: the stream-ordered C entry points on device
buffers (``bfp._lib.call``), and ``bfp.model.BfpModel`` on host arrays.

``listed()`` names the cases, ``draw(rng)`` gives more of the same ranges,
``prepare`` / ``run`` set one up and make one pass, ``work`` is what a pass
cannot do without, ``tolerance`` what another correct implementation may
differ by, and ``exact`` the results in plain 64-bit torch.

Inputs follow the distributions the reference simulator works on: weights
N(0, 0.02) in float32, gammas 1 + N(0, 0.05), activations N(0, 1).
"""
import math
import sys
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "tinyllm-fpga_amd"))

TILE = 16
HD = 64
# D, query heads, KV heads, FFN: the model shape the benchmark runs, and the
# smaller ones of the tests
SHAPES = {"full": (576, 9, 3, 1536), "mid": (256, 4, 2, 512), "small": (192, 3, 1, 256)}
MATS = ("Wq", "Wk", "Wv", "Wo", "Wg", "Wu", "Wd")


# ------------------------------------------------------------------- cases
def listed():
    return [
        # every function of the simulator once, on one token's vectors: the
        # op-by-op use, where a call's latency is all there is
        {"name": "ops_token", "kind": "ops", "n": 576, "ffn": 1536, "heads": 9, "ctx": 72, "rows": 1},
        # the matvec engine over a set of distinct matrices (the sweep of the
        # benchmark: one launch, every weight read from memory once)
        {"name": "matvec_set", "kind": "matvec", "n_out": 1536, "n_in": 576, "mats": 256},
        # loading: a float32 table quantised into the device layout
        {"name": "quantize_table", "kind": "quantize", "n_out": 49152, "n_in": 576},
        # the single-layer harness: one layer, positions 0..7, one call per
        # position with host buffers
        {"name": "layer_positions", "kind": "layer", "shape": "full", "batch": 1, "ctx": 16, "pos": 0, "n": 8},
        # one layer for a ragged batch of sequences at a short context, two
        # positions (the second reads the cache rows the first wrote)
        {"name": "layer_batch", "kind": "layer", "shape": "full", "batch": 50, "ctx": 136, "pos": 99, "n": 2},
        # the same for a batch at a long context: the attention's side
        {"name": "layer_batch_long", "kind": "layer", "shape": "full", "batch": 16, "ctx": 2048, "pos": 1500, "n": 2},
        # the head on its own: final norm, logits and argmax of several
        # hidden states
        {"name": "head_logits", "kind": "head", "D": 576, "vocab": 49152, "batch": 8},
        # short chat turn at batch 1: 8 prompt tokens, 64 generated
        {"name": "decode_short", "kind": "decode", "shape": "full", "layers": 30, "vocab": 49152, "ctx": 72,
         "batch": 1, "prompt": 8, "gen": 64},
        # long document at batch 1: the prompt is most of the work
        {"name": "prompt_long", "kind": "decode", "shape": "full", "layers": 30, "vocab": 49152, "ctx": 2048,
         "batch": 1, "prompt": 1000, "gen": 24},
        # a handful of users: small odd batch
        {"name": "decode_few", "kind": "decode", "shape": "full", "layers": 30, "vocab": 49152, "ctx": 72,
         "batch": 5, "prompt": 23, "gen": 25},
        # throughput serving: 64 sequences
        {"name": "decode_batch", "kind": "decode", "shape": "full", "layers": 30, "vocab": 49152, "ctx": 136,
         "batch": 64, "prompt": 8, "gen": 24},
        # checking the FPGA: its own arithmetic and token loop, every step's
        # last-layer output kept
        {"name": "rtl_decode", "kind": "rtl", "shape": "full", "layers": 30, "vocab": 49152, "ctx": 32,
         "prompt": 4, "gen": 12},
    ]


def _log_int(rng, lo, hi, step=1):
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / step)) * step
    return min(max(v, lo), hi)


def draw(rng):
    kind = rng.choice(["ops", "matvec", "quantize", "layer", "layer", "head", "decode", "decode", "decode", "rtl"])
    if kind == "ops":
        return {"kind": kind, "n": _log_int(rng, 64, 1728, 64), "ffn": _log_int(rng, 64, 1728, 16),
                "heads": rng.randint(1, 27), "ctx": _log_int(rng, 1, 4096), "rows": _log_int(rng, 1, 64)}
    if kind == "matvec":
        n_out, n_in = _log_int(rng, 16, 49152, 16), _log_int(rng, 64, 3456, 16)
        return {"kind": kind, "n_out": n_out, "n_in": n_in,
                "mats": _log_int(rng, 1, max(1, min(1000, (220 << 20) // (n_out * n_in))))}
    if kind == "quantize":
        n_in = _log_int(rng, 64, 1728, 16)
        return {"kind": kind, "n_out": _log_int(rng, 16, 49152, 16), "n_in": n_in}
    if kind == "layer":
        ctx = _log_int(rng, 16, 2048)
        batch = rng.choice([1, 1, _log_int(rng, 2, 64)])
        batch = min(batch, max(1, 40000 // ctx))
        n = rng.randint(1, 8) if batch == 1 else rng.randint(1, 2)
        return {"kind": kind, "shape": rng.choice(["full", "full", "mid", "small"]), "batch": batch, "ctx": ctx,
                "pos": rng.randint(0, ctx - n), "n": n}
    if kind == "head":
        D = rng.choice([576, 576, 256, 192])
        return {"kind": kind, "D": D, "vocab": _log_int(rng, 1024, 49152, 16), "batch": _log_int(rng, 1, 64)}
    vocab = rng.choice([49152, 8192, 1024])
    if kind == "rtl":
        p, g = rng.randint(1, 8), rng.randint(1, 16)
        return {"kind": kind, "shape": rng.choice(["full", "mid"]), "layers": rng.randint(2, 30), "vocab": vocab,
                "ctx": p + g + rng.randint(0, 16), "prompt": p, "gen": g}
    batch = rng.choice([1, 1, _log_int(rng, 2, 64), _log_int(rng, 2, 64)])
    if batch == 1:
        p, g = _log_int(rng, 1, 960), _log_int(rng, 1, 60)
    else:
        p = min(_log_int(rng, 1, 128), max(1, 1500 // batch))
        g = min(_log_int(rng, 1, 32), max(1, 540 // batch))
    ctx = min(2048, p + g + rng.choice([0, 1, 60, 500]))
    return {"kind": "decode", "shape": rng.choice(["full", "full", "full", "mid"]), "layers": rng.choice([30, 12, 2]),
            "vocab": vocab, "ctx": ctx, "batch": batch, "prompt": p, "gen": g}


# ------------------------------------------------------------------ inputs
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _randn(g, *shape, std=1.0, dtype=torch.float32):
    return torch.randn(*shape, generator=g, device="cuda", dtype=dtype) * std


def _quant(v):
    """Tiles of 16 along the last axis: v ~ m 2^(e-15), 16 mantissas to one
    exponent (float64 in; m float64 whole numbers, e float64)."""
    t = v.double().unflatten(-1, (-1, TILE))
    amax = t.abs().amax(-1)
    e = torch.where(amax > 0, torch.floor(torch.log2(amax.clamp_min(1e-300))) + 1, torch.full_like(amax, -127.0))
    e = e.clamp(-127, 127)
    m = torch.round(torch.ldexp(t, (15 - e).unsqueeze(-1))).clamp(-32768, 32767)
    return m.flatten(-2), e


def _value(m, e):
    return torch.ldexp(m.unflatten(-1, (-1, TILE)), (e - 15).unsqueeze(-1)).flatten(-2)


def _q(v):
    return _value(*_quant(v))


def _host(m, e):
    return m.to(torch.int16).cpu().numpy(), e.to(torch.int8).cpu().numpy()


def _dims(case):
    D, hq, hkv, ffn = SHAPES[case["shape"]]
    return D, hq, hkv, ffn, hkv * HD


def _layer_weights(g, D, KV, ffn):
    rows = {"Wq": (D, D), "Wk": (KV, D), "Wv": (KV, D), "Wo": (D, D), "Wg": (ffn, D), "Wu": (ffn, D), "Wd": (D, ffn)}
    flat = _randn(g, sum(r * c for r, c in rows.values()), std=0.02)
    w, at = {}, 0
    for name, (r, c) in rows.items():
        w[name] = flat[at:at + r * c].view(r, c)
        at += r * c
    w["g1"] = 1.0 + _randn(g, D, std=0.05)
    w["g2"] = 1.0 + _randn(g, D, std=0.05)
    return w


def _model_weights(case, seed):
    D, _, _, ffn, KV = _dims(case)
    g = _gen(seed)
    layers = [_layer_weights(g, D, KV, ffn) for _ in range(case["layers"])]
    embed = _randn(g, case["vocab"], D, std=0.02)
    norm_w = 1.0 + _randn(g, D, std=0.05)
    prompt = torch.randint(0, case["vocab"], (case.get("batch", 1), case["prompt"]), generator=g, device="cuda")
    return layers, embed, norm_w, prompt


def _load(case, layers, embed=None, norm_w=None, batch=1):
    from bfp import Dims
    from bfp.model import BfpModel
    D, hq, hkv, ffn, _ = _dims(case)
    m = BfpModel(Dims(D=D, H_Q=hq, H_KV=hkv, HD=HD, FFN=ffn, NL=len(layers), MAX_CTX=case["ctx"],
                      VOCAB=case.get("vocab", 256)), max_batch=batch)
    for li, lw in enumerate(layers):
        for name, w in lw.items():
            m.load_tensor(name, li, fp32=w.cpu().numpy())
    if embed is not None:
        m.load_tensor("embed", fp32=embed.cpu().numpy())
        m.load_tensor("norm_w", fp32=norm_w.cpu().numpy())
    return m


def _layer_inputs(case, seed):
    """Weights, the calls' inputs (n, batch, D) and the cache's rows before
    them (batch, pos, KV) as (m, e) pairs of float64."""
    D, _, _, ffn, KV = _dims(case)
    g = _gen(seed)
    w = _layer_weights(g, D, KV, ffn)
    h = _quant(_randn(g, case["n"], case["batch"], D, dtype=torch.float64))
    # a cache row is a matvec of a normed hidden: about N(0, 0.02 sqrt(D))
    std = 0.02 * math.sqrt(D)
    k = _quant(_randn(g, case["batch"], case["pos"], KV, std=std, dtype=torch.float64))
    v = _quant(_randn(g, case["batch"], case["pos"], KV, std=std, dtype=torch.float64))
    return w, h, k, v


def _ops_inputs(case, seed):
    g = _gen(seed)
    n, ffn, heads, ctx, rows = (case[k] for k in ("n", "ffn", "heads", "ctx", "rows"))
    f64 = torch.float64
    return {"v": _randn(g, rows * n, dtype=f64), "W": _randn(g, n, n, std=0.02),
            "x": _q(_randn(g, rows, n, dtype=f64)), "gamma": _q(1.0 + _randn(g, n, std=0.05, dtype=f64)),
            "gate": _q(_randn(g, rows, ffn, dtype=f64)), "scores": _randn(g, rows * heads, ctx, dtype=f64),
            "q": _q(_randn(g, rows * heads, HD, dtype=f64)), "pos": case["ctx"] - 1}


# ----------------------------------------------------------------- prepare
def prepare(case, seed):
    kind = case["kind"]
    if kind == "ops":
        from bfp._lib import call
        i = _ops_inputs(case, seed)
        rows, n = case["rows"], case["n"]
        cs = np.empty(HD, np.float64)
        call("bfp_rope_cos_sin", i["pos"], HD, 10000.0, cs.ctypes.data)
        Pm, Pe = _packed(i["W"][None])
        dev = {"device": "cuda"}
        out = {"m": torch.empty(rows * n, dtype=torch.int16, **dev),
               "e": torch.empty(rows * n // TILE, dtype=torch.int8, **dev),
               "ym": torch.empty(rows * n, dtype=torch.int16, **dev),
               "ye": torch.empty(rows * n // TILE, dtype=torch.int8, **dev),
               "y": torch.empty(rows, n, dtype=torch.float64, **dev), "norm": torch.empty_like(i["x"]),
               "silu": torch.empty_like(i["gate"]), "soft": torch.empty_like(i["scores"]),
               "rope": torch.empty_like(i["q"])}
        return {"case": case, "i": i, "cs": torch.from_numpy(cs).cuda(), "P": (Pm, Pe), "out": out}
    if kind == "matvec":
        g = _gen(seed)
        Pm, Pe = _packed(_randn(g, case["mats"], case["n_out"], case["n_in"], std=0.02))
        xm, xe = _quant(_randn(g, case["mats"], case["n_in"], dtype=torch.float64))
        ym = torch.empty(case["mats"], case["n_out"], dtype=torch.int16, device="cuda")
        ye = torch.empty(case["mats"], case["n_out"] // TILE, dtype=torch.int8, device="cuda")
        return {"case": case, "P": (Pm, Pe), "x": (xm.to(torch.int16), xe.to(torch.int8)), "y": (ym, ye)}
    if kind == "quantize":
        W = _randn(_gen(seed), case["n_out"], case["n_in"], std=0.02)
        n = W.numel()
        return {"case": case, "W": W, "P": (torch.empty(n, dtype=torch.int16, device="cuda"),
                                            torch.empty(n // TILE, dtype=torch.int8, device="cuda"))}
    if kind == "layer":
        w, h, k, v = _layer_inputs(case, seed)
        m = _load(case, [w], batch=case["batch"])
        if case["pos"]:
            km, ke = _host(*k)
            vm, ve = _host(*v)
            for b in range(case["batch"]):
                m.kv_io(0, b, 0, case["pos"], k=(km[b], ke[b]), v=(vm[b], ve[b]))
        return {"case": case, "model": m, "h": _host(*h)}
    if kind == "head":
        m, hm, he = _head_model(case, seed)
        return {"case": case, "model": m, "h": (hm, he)}
    layers, embed, norm_w, prompt = _model_weights(case, seed)
    m = _load(case, layers, embed, norm_w, batch=case.get("batch", 1))
    return {"case": case, "model": m, "prompt": prompt.to(torch.int32).cpu().numpy()}


def _packed(W):
    """quantize_W of (mats, n_out, n_in) float32 matrices into the device
    layout, matrix after matrix."""
    from bfp._lib import call
    mats, n_out, n_in = W.shape
    Pm = torch.empty(mats, n_out * n_in, dtype=torch.int16, device="cuda")
    Pe = torch.empty(mats, n_out * n_in // TILE, dtype=torch.int8, device="cuda")
    s = torch.cuda.current_stream().cuda_stream
    for k in range(mats):
        call("bfp_quantize_pack_f32_d", W[k].data_ptr(), n_out, n_in, Pm[k].data_ptr(), Pe[k].data_ptr(), s)
    torch.cuda.synchronize()
    return Pm, Pe


def _head_inputs(case, seed):
    g = _gen(seed)
    h = _quant(_randn(g, case["batch"], case["D"], dtype=torch.float64))
    return h, _randn(g, case["vocab"], case["D"], std=0.02), 1.0 + _randn(g, case["D"], std=0.05)


def _head_model(case, seed):
    from bfp import Dims
    from bfp.model import BfpModel
    h, embed, norm_w = _head_inputs(case, seed)
    D = case["D"]
    m = BfpModel(Dims(D=D, H_Q=D // HD, H_KV=1, HD=HD, FFN=256, NL=1, MAX_CTX=16, VOCAB=case["vocab"]),
                 max_batch=case["batch"])
    m.load_tensor("embed", fp32=embed.cpu().numpy())
    m.load_tensor("norm_w", fp32=norm_w.cpu().numpy())
    return (m, *_host(*h))


# --------------------------------------------------------------------- run
def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "ops":
        return _run_ops(state)
    if kind == "matvec":
        from bfp._lib import call
        (Pm, Pe), (xm, xe), (ym, ye) = state["P"], state["x"], state["y"]
        n_out, n_in = case["n_out"], case["n_in"]
        call("bfp_matvec_d", Pm.data_ptr(), Pe.data_ptr(), n_out, n_in, case["mats"], n_out * n_in * 2,
             n_out * n_in // TILE, xm.data_ptr(), xe.data_ptr(), n_in, ym.data_ptr(), ye.data_ptr(), n_out, 0,
             torch.cuda.current_stream().cuda_stream)
        return ym, ye
    if kind == "quantize":
        from bfp._lib import call
        W, (Pm, Pe) = state["W"], state["P"]
        call("bfp_quantize_pack_f32_d", W.data_ptr(), case["n_out"], case["n_in"], Pm.data_ptr(), Pe.data_ptr(),
             torch.cuda.current_stream().cuda_stream)
        return Pm, Pe
    m = state["model"]
    if kind == "layer":
        hm, he = state["h"]
        return [m.layer_step_bfp(0, case["pos"] + j, hm[j], he[j])[:2] for j in range(case["n"])]
    if kind == "head":
        return m.head(*state["h"], logits=True)
    if kind == "rtl":
        preds, hist = m.rtl_decode(state["prompt"][0], case["gen"], hist=True)
        return preds, hist
    # every layer's output at every step beside the tokens, and the last
    # step's logits from the head
    toks, (hm, he) = m.decode(state["prompt"], case["gen"], hist=True)
    last, logits = m.head(hm[:, -1, -1], he[:, -1, -1], logits=True)
    return toks, hm, he, last, logits


def _run_ops(state):
    from bfp._lib import call
    case, i, o = state["case"], state["i"], state["out"]
    Pm, Pe = state["P"]
    s = torch.cuda.current_stream().cuda_stream
    n, ffn, heads, ctx, rows = (case[k] for k in ("n", "ffn", "heads", "ctx", "rows"))
    call("bfp_tile_quantize_f64_d", i["v"].data_ptr(), rows * n, o["m"].data_ptr(), o["e"].data_ptr(), s)
    # one matrix, `rows` input vectors
    call("bfp_matvec_ring_d", Pm.data_ptr(), Pe.data_ptr(), n, n, rows, 1, 0, 0, o["m"].data_ptr(),
         o["e"].data_ptr(), n, o["ym"].data_ptr(), o["ye"].data_ptr(), n, 0, s)
    call("bfp_tile_decode_d", o["ym"].data_ptr(), o["ye"].data_ptr(), rows * n, o["y"].data_ptr(), s)
    call("bfp_rmsnorm_fp_d", i["x"].data_ptr(), i["gamma"].data_ptr(), n, rows, 1e-5, o["norm"].data_ptr(), s)
    call("bfp_silu_fp_d", i["gate"].data_ptr(), rows * ffn, o["silu"].data_ptr(), s)
    call("bfp_softmax_fp_d", i["scores"].data_ptr(), ctx, rows * heads, o["soft"].data_ptr(), s)
    call("bfp_rope_fp_d", i["q"].data_ptr(), rows * heads, state["cs"].data_ptr(), o["rope"].data_ptr(), s)
    return [o[k] for k in ("m", "e", "ym", "ye", "y", "norm", "silu", "soft", "rope")]


# -------------------------------------------------------------------- work
def _layer_params(case):
    D, _, _, ffn, KV = _dims(case)
    return (2 * D + 2 * KV) * D + 3 * D * ffn


def _bfp_bytes(n):
    return n * 2 + n // TILE


def work(case):
    """Bytes: each weight, cache row, input and output once for every call
    that cannot share it with another (a prompt's positions can share one
    reading of the weights; generated tokens follow one another)."""
    kind = case["kind"]
    if kind == "ops":
        n, ffn, heads, ctx, rows = (case[k] for k in ("n", "ffn", "heads", "ctx", "rows"))
        b = rows * (n * 8 + _bfp_bytes(n)) + _bfp_bytes(n * n) + rows * (_bfp_bytes(n) + n * 8)
        b += rows * n * 16 + n * 8 + rows * ffn * 16 + rows * heads * (ctx + HD) * 16 + HD * 8
        return {"bytes": b, "flops": rows * (2 * n * n + 10 * (n + ffn + heads * (ctx + HD)))}
    if kind == "matvec":
        n_out, n_in, mats = case["n_out"], case["n_in"], case["mats"]
        return {"bytes": mats * (_bfp_bytes(n_out * n_in) + _bfp_bytes(n_in) + _bfp_bytes(n_out)),
                "flops": 2 * mats * n_out * n_in}
    if kind == "quantize":
        n = case["n_out"] * case["n_in"]
        return {"bytes": n * 4 + _bfp_bytes(n), "flops": 3 * n}
    if kind == "head":
        b, v, D = case["batch"], case["vocab"], case["D"]
        return {"bytes": v * D * 4 + b * v * 8 + b * _bfp_bytes(D), "flops": 2 * b * v * D}
    D, hq, _, _, KV = _dims(case)
    P = _layer_params(case)
    if kind == "layer":
        B, p, n = case["batch"], case["pos"], case["n"]
        ctx = sum(p + j for j in range(n))
        return {"bytes": n * _bfp_bytes(P) + B * (2 * ctx * _bfp_bytes(KV) + n * 2 * _bfp_bytes(KV + D)),
                "flops": 2 * B * (n * P + 2 * hq * HD * (ctx + n))}
    L, V, p, g = case["layers"], case["vocab"], case["prompt"], case["gen"]
    B = case.get("batch", 1)
    steps = p + g
    heads = steps if kind == "rtl" else g + 1
    cached = sum(range(p, steps)) + p            # cache rows read: per generated step, once for the prompt
    hist = steps * (1 if kind == "rtl" else L) * _bfp_bytes(D)
    emb = _bfp_bytes(V * D) if kind == "rtl" else V * D * 4
    return {"bytes": (g + 1) * L * _bfp_bytes(P) + (g + 1) * emb + B * (2 * L * (cached + steps) * _bfp_bytes(KV) + hist),
            "flops": 2 * B * (steps * L * P + heads * V * D + 2 * L * hq * HD * sum(range(1, steps + 1)))}


# --------------------------------------------------------------- tolerance
def tolerance(case):
    """BFP results are whole numbers that the format defines exactly, so
    they have to be equal.  Only softmax_fp's probabilities (another
    correctly working exp or order of the sum: measured 1.1e-16 from
    torch's) and the logits (another order of a 576-term float64 sum:
    measured 8.7e-16) leave the kernels as float64."""
    if case["kind"] == "ops":
        return {"rel": 5e-16, "max": 1e-14, "differ": 0.0}
    if case["kind"] in ("head", "decode"):
        return {"rel": 4e-15, "max": 1e-13, "differ": 0.0}
    return "exact"


# ------------------------------------------------------------------- exact
def _matvec64(x, Wm, We):
    """The engine's matvec in float64 whole numbers: x (..., in) float64
    values, W (out, in) tiles -> (m, e).  Tile sums are exact (below 2^35),
    aligned to the row's largest exponent with a floor, dropped past 47
    bits."""
    xm, xe = _quant(x)
    lead = xm.shape[:-1]
    xm, xe = xm.reshape(-1, xm.shape[-1]), xe.reshape(-1, xe.shape[-1])
    nT = xe.shape[-1]
    out = []
    rows = max(TILE, (1 << 26) // (xm.shape[0] * nT) // TILE * TILE)
    for r in range(0, Wm.shape[0], rows):
        W = Wm[r:r + rows].unflatten(-1, (nT, TILE))
        S = torch.einsum("btk,otk->bot", xm.unflatten(-1, (nT, TILE)), W) if xm.shape[0] == 1 else \
            torch.bmm(xm.unflatten(-1, (nT, TILE)).transpose(0, 1).contiguous(),
                      W.permute(1, 2, 0).contiguous()).permute(1, 2, 0)
        E = xe.unsqueeze(1) + We[r:r + rows].unsqueeze(0)
        M = E.amax(-1, keepdim=True)
        d = M - E
        A = torch.where(d <= 47, torch.floor(torch.ldexp(S, -d)), torch.zeros_like(S)).sum(-1)
        out.append(torch.ldexp(A.clamp(-2.0 ** 47, 2.0 ** 47 - 1), M.squeeze(-1) - 30))
    return _quant(torch.cat(out, -1).reshape(*lead, -1))


def _rms64(x, gamma):
    return (x * gamma) / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-5)


def _rope64(x, pos):
    """x (..., heads, 64) at positions pos (broadcast over the lead axes)."""
    j = torch.arange(HD // 2, device="cuda", dtype=torch.float64)
    th = (1.0 / (10000.0 ** (2 * j / HD))) * pos.unsqueeze(-1)
    c, s = torch.cos(th), torch.sin(th)
    a, b = x[..., :HD // 2], x[..., HD // 2:]
    return torch.cat([a * c - b * s, b * c + a * s], -1)


class _Layer64:
    """One decoder layer on float64 values, every stage in BFP."""

    def __init__(self, case, w):
        _, self.hq, self.hkv, _, _ = _dims(case)
        self.W = {k: _quant(w[k]) for k in MATS}
        self.g1, self.g2 = _q(w["g1"]), _q(w["g2"])

    def mv(self, x, name):
        return _value(*_matvec64(x, *self.W[name]))

    def __call__(self, h, K, V, p0):
        """h (B, n, D): positions p0 .. p0+n-1 of each sequence; K, V (B, T,
        hkv, 64) hold the rows before p0 and take the new ones."""
        B, n, D = h.shape
        pos = torch.arange(p0, p0 + n, device="cuda", dtype=torch.float64)
        x = _rms64(h, self.g1)
        x = _q(x)
        q = self.mv(x, "Wq").view(B, n, self.hq, HD)
        k = self.mv(x, "Wk").view(B, n, self.hkv, HD)
        q, k = (_q(_rope64(t, pos.view(1, n, 1))) for t in (q, k))
        K[:, p0:p0 + n] = k
        V[:, p0:p0 + n] = self.mv(x, "Wv").view(B, n, self.hkv, HD)
        T = p0 + n
        grp = self.hq // self.hkv
        att = torch.empty(B, n, self.hq, HD, dtype=torch.float64, device="cuda")
        mask = torch.arange(T, device="cuda").view(1, T) > torch.arange(p0, T, device="cuda").view(n, 1)
        for a in range(self.hq):
            Kt = K[:, :T, a // grp].transpose(1, 2).contiguous()
            s = torch.bmm(q[:, :, a].contiguous(), Kt) / 8.0
            p = torch.softmax(s.masked_fill(mask, -torch.inf), -1)
            att[:, :, a] = torch.bmm(p, V[:, :T, a // grp].contiguous())
        o = self.mv(_q(att.view(B, n, D)), "Wo")
        h1 = _q(h + o)
        x = _q(_rms64(h1, self.g2))
        gate, up = self.mv(x, "Wg"), self.mv(x, "Wu")
        mlp = _q(_q(gate / (1.0 + torch.exp(-gate))) * up)
        return h1 + self.mv(mlp, "Wd")


def _logits64(h, embed, norm_w):
    hn = (h / torch.sqrt((h * h).mean(-1, keepdim=True) + 1e-5)) * norm_w
    return hn @ embed.double().t()


def exact(case, seed):
    kind = case["kind"]
    if kind == "ops":
        i = _ops_inputs(case, seed)
        m, e = _quant(i["v"])
        Wm, We = _quant(i["W"])
        ym, ye = _matvec64(_value(m, e).view(case["rows"], case["n"]), Wm, We)
        pos = torch.tensor(float(i["pos"]), dtype=torch.float64, device="cuda")
        return [m, e, ym.flatten(), ye.flatten(), _value(ym, ye), _q(_rms64(i["x"], i["gamma"])),
                _q(i["gate"] / (1.0 + torch.exp(-i["gate"]))), torch.softmax(i["scores"], -1),
                _q(_rope64(i["q"], pos))]
    if kind == "matvec":
        g = _gen(seed)
        W = _randn(g, case["mats"], case["n_out"], case["n_in"], std=0.02)
        x = _randn(g, case["mats"], case["n_in"], dtype=torch.float64)
        ym, ye = zip(*(_matvec64(_q(x[k])[None], *_quant(W[k])) for k in range(case["mats"])))
        return torch.cat(ym), torch.cat(ye)
    if kind == "quantize":
        W = _randn(_gen(seed), case["n_out"], case["n_in"], std=0.02)
        m, e = _quant(W)
        nT = case["n_in"] // TILE
        # the device layout: 16-row chunks, tile-major, two 8-column halves
        m = m.view(-1, 16, nT, 2, 8).permute(0, 2, 3, 1, 4).flatten()
        return m.to(torch.int16), e.view(-1, 16, nT).permute(0, 2, 1).flatten().to(torch.int8)
    if kind == "layer":
        w, h, k, v = _layer_inputs(case, seed)
        _, _, hkv, _, _ = _dims(case)
        p, n, B = case["pos"], case["n"], case["batch"]
        K = torch.zeros(B, p + n, hkv, HD, dtype=torch.float64, device="cuda")
        V = torch.zeros_like(K)
        if p:
            K[:, :p] = _value(*k).view(B, p, hkv, HD)
            V[:, :p] = _value(*v).view(B, p, hkv, HD)
        layer, hv = _Layer64(case, w), _value(*h)
        out = [_quant(layer(hv[j][:, None], K, V, p + j)[:, 0]) for j in range(n)]
        return [_host(*o) for o in out]
    if kind == "head":
        h, embed, norm_w = _head_inputs(case, seed)
        lg = _logits64(_value(*h), embed, _q(norm_w))
        return lg.argmax(-1).to(torch.int32).cpu().numpy(), lg.cpu().numpy()
    if kind == "rtl":
        return None          # the FPGA's truncating integer engines: no 64-bit value
    if (case["prompt"] + case["gen"]) * case["layers"] > 2500 or case["batch"] * (case["prompt"] + case["gen"]) > 3000:
        return None          # step by step in plain torch: too long
    return _decode64(case, seed)


def _decode64(case, seed):
    weights, embed, norm_w, prompt = _model_weights(case, seed)
    D, _, hkv, _, _ = _dims(case)
    B, p, g = case["batch"], case["prompt"], case["gen"]
    layers = [_Layer64(case, w) for w in weights]
    norm = _q(norm_w)
    K = [torch.zeros(B, p + g, hkv, HD, dtype=torch.float64, device="cuda") for _ in layers]
    V = [torch.zeros_like(k) for k in K]
    hist = torch.zeros(B, p + g, len(layers), D, dtype=torch.float64, device="cuda")
    toks = []

    def step(ids, p0):
        h = _q(embed[ids].double())
        for li, layer in enumerate(layers):
            h = _q(layer(h, K[li], V[li], p0))
            hist[:, p0:p0 + h.shape[1], li] = h
        return h[:, -1]

    step(prompt, 0)
    ids = prompt[:, -1:]          # the loop feeds the last prompt token once more
    for s in range(g):
        ids = _logits64(step(ids, p + s), embed, norm).argmax(-1, keepdim=True)
        toks.append(ids)
    hm, he = _host(*_quant(hist))
    lg = _logits64(_value(*_quant(hist[:, -1, -1])), embed, norm)
    return (torch.cat(toks, 1).to(torch.int32).cpu().numpy(), hm, he,
            lg.argmax(-1).to(torch.int32).cpu().numpy(), lg.cpu().numpy())
