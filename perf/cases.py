"""What this framework's speed is measured on: the calls that a program
serving a 4-bit Qwen2-architecture model makes, from the smallest (the
activation codec of one decode step) to the largest (the whole decode sweep).

The listed sizes are those of the repository's own 7B configuration
(hetero/qwen2.py: hidden 3584, intermediate 18944, 28 query heads and 4 KV
heads of 128, vocabulary 152064, group size 64); draw() spreads the same
calls over other widths, row counts, contexts and options.  Run with the
repository's root as the working folder.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.getcwd(), "hetero-infer_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from hetero import gpu_model, q4, qlinear, qwen2, sweep, transport  # noqa: E402

HIDDEN, INTER, HEADS, KV_HEADS, HEAD_DIM, VOCAB = 3584, 18944, 28, 4, 128, 152064


# ---- the cases ---------------------------------------------------------------

def listed():
    return [
        # a pipeline stage hands the hidden state of one decoded token to the next stage
        {"name": "wire_one_token", "kind": "wire", "codec": "int8", "rows": 1, "hidden": HIDDEN},
        # the reference's NumPy backend with this library dropped in: one projection of one
        # token on host arrays, through the C interface
        {"name": "dropin_linear", "kind": "dropin", "rows": 1, "n_out": HIDDEN, "n_in": HIDDEN, "gs": 64},
        # one decoder layer of a decode step at a 2048-token context, captured in a HIP graph
        # as the device-resident stage captures its steps
        {"name": "decode_layer", "kind": "layer", "hidden": HIDDEN, "inter": INTER, "heads": HEADS,
         "kv_heads": KV_HEADS, "head_dim": HEAD_DIM, "context": 2048},
        # the attention of one decoded token deep in a long conversation
        {"name": "decode_attention_long", "kind": "decode_attention", "heads": HEADS, "kv_heads": KV_HEADS,
         "head_dim": HEAD_DIM, "context": 12345},
        # the MLP block of a few rows: small decode batches, speculative verification
        {"name": "mlp_5_rows", "kind": "mlp", "rows": 5, "hidden": HIDDEN, "inter": INTER, "gs": 64},
        # the grouped q/k/v projections at the most rows that take the GEMV path
        {"name": "qkv_16_rows", "kind": "linear", "rows": 16, "n_in": HIDDEN, "n_out": "3584,512,512", "gs": 64},
        # the grouped q/k/v projections of a short prompt (or the ragged last chunk of a long one)
        {"name": "prompt_qkv_37_rows", "kind": "prompt_linear", "rows": 37, "n_in": HIDDEN, "n_out": "3584,512,512",
         "x_bf16": False},
        # the MLP block of a full prompt chunk
        {"name": "prompt_mlp_512_rows", "kind": "prompt_mlp", "rows": 512, "hidden": HIDDEN, "inter": INTER},
        # the causal attention of the fourth chunk of a 2048-token prompt
        {"name": "prompt_attention_512", "kind": "prompt_attention", "rows": 512, "context": 1536, "heads": HEADS,
         "kv_heads": KV_HEADS, "head_dim": HEAD_DIM, "out_bf16": False},
        # the headline benchmark: all projections of a decode step as one chained program
        {"name": "decode_sweep", "kind": "sweep", "layers": 28, "hidden": HIDDEN, "inter": INTER, "vocab": VOCAB},
        # one token through the whole device-resident model
        {"name": "decode_step", "kind": "step", "layers": 28, "context": 2048, "vocab": VOCAB},
        # a 512-token prompt through a device-resident stage of three layers and the head (a
        # pipeline stage's share; more layers only repeat the same calls)
        {"name": "prefill_3_layers", "kind": "prefill", "layers": 3, "rows": 512, "context": 0, "vocab": VOCAB},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _width(rng, lo, hi, step):
    """A multiple of step in [lo, hi], spread over its logarithm."""
    return max(lo // step, min(hi // step, int(round(_log_int(rng, lo, hi) / step)))) * step


def _heads(rng):
    kv = rng.choice([2, 4, 8])
    group = rng.choice([1, 2, 4, 7, 8])
    return {"heads": kv * group, "kv_heads": kv, "head_dim": rng.choice([128, 128, 128, 64])}


def draw(rng):
    kind = rng.choice(["wire", "dropin", "layer", "decode_attention", "mlp", "linear", "prompt_linear", "prompt_mlp",
                       "prompt_attention", "sweep", "step", "prefill"])
    c = {"kind": kind}
    if kind == "wire":
        c.update(codec=rng.choice(["int8", "fp16"]), rows=_log_int(rng, 1, 2048),
                 hidden=rng.choice([_width(rng, 896, 8192, 128), _log_int(rng, 500, 8192)]))
    elif kind == "dropin":
        c.update(rows=_log_int(rng, 1, 16), n_out=_log_int(rng, 256, 19000), n_in=_width(rng, 512, 18944, 128),
                 gs=rng.choice([64, 64, 128]))
    elif kind == "layer":
        c.update(_heads(rng))
        c["head_dim"] = 128
        c.update(hidden=c["heads"] * 128, inter=_width(rng, 2048, 18944, 128), context=_log_int(rng, 1, 8192))
    elif kind == "decode_attention":
        c.update(_heads(rng), context=_log_int(rng, 16, 32768))
    elif kind == "mlp":
        c.update(rows=rng.randint(1, 16), hidden=_width(rng, 896, 5120, 128), inter=_width(rng, 4864, 18944, 128),
                 gs=rng.choice([64, 64, 64, 128]))
    elif kind == "linear":
        n = rng.choice([1, 1, 2, 3])
        c.update(rows=rng.randint(1, 16), n_in=_width(rng, 896, 18944, 128),
                 n_out=",".join(str(_log_int(rng, 200, 19000)) for _ in range(n)), gs=rng.choice([64, 64, 64, 128]))
    elif kind == "prompt_linear":
        n = rng.choice([1, 1, 2, 3])
        c.update(rows=_log_int(rng, 17, 1024), n_in=_width(rng, 896, 18944, 64),
                 n_out=",".join(str(_log_int(rng, 200, 19000)) for _ in range(n)), x_bf16=rng.choice([False, True]))
    elif kind == "prompt_mlp":
        c.update(rows=_log_int(rng, 17, 1024), hidden=_width(rng, 896, 5120, 64), inter=_width(rng, 4864, 18944, 64))
    elif kind == "prompt_attention":
        c.update(_heads(rng), rows=_log_int(rng, 2, 768), context=rng.choice([0, _log_int(rng, 16, 6144)]),
                 out_bf16=rng.choice([False, True]))
    elif kind == "sweep":
        c.update(layers=rng.randint(1, 27), hidden=_width(rng, 1024, 3584, 128), inter=_width(rng, 4864, 18944, 128),
                 vocab=_log_int(rng, 30000, VOCAB))
    elif kind == "step":
        c.update(layers=rng.randint(2, 20), context=_log_int(rng, 16, 6144), vocab=_log_int(rng, 30000, VOCAB))
    else:
        c.update(layers=rng.randint(1, 3), rows=_log_int(rng, 2, 700), context=rng.choice([0, 0, _log_int(rng, 16, 1024)]),
                 vocab=_log_int(rng, 30000, VOCAB))
    return c


# ---- inputs ------------------------------------------------------------------

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 7919 + 17)
    return g


def _mat(g, n_out, n_in, gs=64, center=7.5):
    """A packed 4-bit matrix: uniform nibbles, fp16 scales |N(0, 0.02)| * sqrt(1024 / n_in) and biases that centre
    the dequantised values near zero, as trained weights are."""
    w = torch.randint(-2**31, 2**31, (n_out, n_in // 8), dtype=torch.int64, device="cuda", generator=g).to(torch.int32)
    s = (torch.randn((n_out, n_in // gs), device="cuda", generator=g) * 0.02 * math.sqrt(1024 / n_in)).abs().half()
    b = (-center * s.float() + torch.randn(s.shape, device="cuda", generator=g) * 0.002).half()
    return w, s.view(torch.int16), b.view(torch.int16)


def _randn(g, *shape):
    return torch.randn(shape, device="cuda", generator=g)


def _outs(case):
    return [int(n) for n in case["n_out"].split(",")]


def _cfg(case):
    cfg = qwen2.qwen2_7b_config(case["layers"])
    cfg["vocab_size"] = case["vocab"]
    return cfg


def _weights(cfg, g):
    out = {}
    for name, kind, shape in qwen2.tensor_specs(cfg):
        if kind == "q4":
            w, s, b = _mat(g, *shape)
            out[f"{name}.weight"] = w
            out[f"{name}.scales"], out[f"{name}.biases"] = s.view(torch.float16), b.view(torch.float16)
        else:
            out[name] = _randn(g, *shape) * 0.02 + (1.0 if kind == "norm" else 0.0)
    return out


def _rope(positions, dim):
    inv = 1e6 ** (-np.arange(0, dim // 2, dtype=np.float32) * 2.0 / dim)
    ang = np.arange(positions, dtype=np.float32)[:, None] * inv[None, :]
    return torch.from_numpy(np.cos(ang)).cuda(), torch.from_numpy(np.sin(ang)).cuda()


def _kv(g, kv_heads, cap, dim, held):
    """A key/value cache pair of capacity cap, `held` positions filled."""
    out = []
    for _ in range(2):
        c = torch.zeros((kv_heads, cap, dim), dtype=torch.float16, device="cuda")
        if held:
            c[:, :held] = _randn(g, kv_heads, held, dim).half()
        out.append(c)
    return out


def _attention_inputs(case, g, hidden=None):
    h, kv, d, ctx = case["heads"], case["kv_heads"], case["head_dim"], case["context"]
    cap = (ctx // 256 + 1) * 256
    lib = q4.load()
    s = {"lib": lib, "cap": cap, "scale": float(np.float32(d ** -0.5))}
    s["cos"], s["sin"] = _rope(cap, d)
    s["k_cache"], s["v_cache"] = _kv(g, kv, cap, d, ctx)
    s["bias"] = _randn(g, (h + 2 * kv) * d) * 0.02
    s["pos"] = torch.full((1,), ctx, dtype=torch.int64, device="cuda")
    s["scratch"] = torch.zeros(lib.q4_attention_scratch_floats(h, d, cap), device="cuda")
    s["attn"] = torch.zeros((1, h * d), device="cuda")
    return s


def _decode_attention(case, s, q, k, v):
    lib = s["lib"]
    p = lambda t: t.data_ptr()
    q4.check(lib, lib.q4_attention_rope_dev(
        p(q), p(k), p(v), p(s["bias"]), p(s["cos"]), p(s["sin"]), p(s["pos"]), p(s["k_cache"]), p(s["v_cache"]),
        p(s["attn"]), p(s["scratch"]), case["heads"], case["kv_heads"], case["head_dim"], s["cap"], s["scale"],
        torch.cuda.current_stream().cuda_stream), "attention")


def _layer_calls(case, s):
    q4.norm_gemv_multi_dev(s["qkv"], s["x"], s["delta"], s["in_w"], 1e-6, x_out=s["x1"],
                           outs=[s["q"], s["k"], s["v"]])
    _decode_attention(case, s, s["q"], s["k"], s["v"])
    q4.gemv_dev(*s["o"], s["attn"], out=s["o_out"])
    q4.norm_gate_up_silu_dev(s["gate"], s["up"], s["x1"], s["o_out"], s["post_w"], 1e-6, x_out=s["x2"], h=s["h"])
    q4.gemv_dev(*s["down"], s["h"], out=s["mlp_out"])


def _sweep_shapes(case):
    h, i = case["hidden"], case["inter"]
    kv = h // 7 if h % 448 == 0 else h // 4
    kv = (kv + 7) // 8 * 8
    return [[(h, h), (kv, h), (kv, h)], [(h, h)], [(i, h), (i, h)], [(h, i)]], (case["vocab"], h)


def prepare(case, seed):
    g = _gen(seed)
    kind = case["kind"]
    st = {"case": case}
    if kind == "wire":
        st["x"] = _randn(g, case["rows"], case["hidden"]) * 3.0
    elif kind == "dropin":
        w, s, b = _mat(g, case["n_out"], case["n_in"], case["gs"])
        st["op"] = qlinear.QLinear(w.cpu().numpy().view(np.uint32), s.cpu().numpy().view(np.float16),
                                   b.cpu().numpy().view(np.float16), None, case["gs"], 4)
        st["x"] = _randn(g, case["rows"], case["n_in"]).cpu().numpy()
    elif kind == "layer":
        h, i, d = case["hidden"], case["inter"], case["head_dim"]
        kvd = case["kv_heads"] * d
        st.update(_attention_inputs(case, g))
        st["qkv"] = [_mat(g, n, h) for n in (h, kvd, kvd)]
        st["o"], st["gate"], st["up"], st["down"] = _mat(g, h, h), _mat(g, i, h), _mat(g, i, h), _mat(g, h, i)
        st["in_w"], st["post_w"] = _randn(g, h) * 0.02 + 1.0, _randn(g, h) * 0.02 + 1.0
        st["x"], st["delta"] = _randn(g, h), _randn(g, h)
        for name, n in (("x1", h), ("x2", h), ("q", h), ("k", kvd), ("v", kvd), ("o_out", h), ("h", i),
                        ("mlp_out", h)):
            st[name] = torch.zeros((1, n), device="cuda")
        stream = torch.cuda.Stream()
        stream.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(stream):
            _layer_calls(case, st)
        torch.cuda.synchronize()
        st["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(st["graph"], stream=stream):
            _layer_calls(case, st)
    elif kind == "decode_attention":
        st.update(_attention_inputs(case, g))
        d = case["head_dim"]
        for name, n in (("q", case["heads"] * d), ("k", case["kv_heads"] * d), ("v", case["kv_heads"] * d)):
            st[name] = _randn(g, 1, n)
    elif kind == "mlp":
        h, i, gs, m = case["hidden"], case["inter"], case["gs"], case["rows"]
        st["gate"], st["up"], st["down"] = _mat(g, i, h, gs), _mat(g, i, h, gs), _mat(g, h, i, gs)
        st["x"], st["h"], st["out"] = _randn(g, m, h), torch.zeros((m, i), device="cuda"), torch.zeros((m, h), device="cuda")
    elif kind in ("linear", "prompt_linear"):
        gs, m = case.get("gs", 64), case["rows"]
        st["mats"] = [_mat(g, n, case["n_in"], gs) for n in _outs(case)]
        st["x"] = _randn(g, m, case["n_in"])
        if case.get("x_bf16"):
            st["x"] = st["x"].bfloat16()
        st["outs"] = [torch.zeros((m, n), device="cuda") for n in _outs(case)]
    elif kind == "prompt_mlp":
        h, i, m = case["hidden"], case["inter"], case["rows"]
        st["gate"], st["up"], st["down"] = _mat(g, i, h), _mat(g, i, h), _mat(g, h, i)
        st["x"] = _randn(g, m, h).bfloat16()
        st["h"] = torch.zeros((m, i), dtype=torch.bfloat16, device="cuda")
        st["out"] = torch.zeros((m, h), device="cuda")
    elif kind == "prompt_attention":
        d, rows, ctx = case["head_dim"], case["rows"], case["context"]
        st["lib"] = q4.load()
        st["cap"] = ((ctx + rows) // 256 + 1) * 256
        st["k_cache"], st["v_cache"] = _kv(g, case["kv_heads"], st["cap"], d, ctx + rows)
        st["q"] = _randn(g, rows, case["heads"] * d)
        st["out"] = torch.zeros((rows, case["heads"] * d), device="cuda",
                                dtype=torch.bfloat16 if case["out_bf16"] else torch.float32)
        st["scale"] = float(np.float32(d ** -0.5))
    elif kind == "sweep":
        layer, head = _sweep_shapes(case)
        xs = {n: _randn(g, 1, n) for n in sorted({case["hidden"], case["inter"]})}
        shapes = layer * case["layers"] + [[head]]
        # every output in one buffer, each starting at a 16-byte boundary
        total = sum((n + 3) // 4 * 4 for ph in shapes for n, _ in ph)
        st["out"] = torch.zeros(total, device="cuda")
        phases, at = [], 0
        for ph in shapes:
            mats = [_mat(g, n, k) for n, k in ph]
            outs = []
            for n, _ in ph:
                outs.append(st["out"][at:at + n])
                at += (n + 3) // 4 * 4
            phases.append((mats, xs[ph[0][1]], outs, False))
        st["phases"] = phases
        st["chain"] = q4.Chain(phases)
    elif kind in ("step", "prefill"):
        cfg = _cfg(case)
        w = _weights(cfg, g)
        ctx = case["context"]
        kv = [(_randn(g, KV_HEADS, ctx, HEAD_DIM).half(), _randn(g, KV_HEADS, ctx, HEAD_DIM).half())
              for _ in range(case["layers"])] if ctx else None
        st["stage"] = gpu_model.GpuStage(cfg, w, None if kv is None else [a for a, _ in kv],
                                         None if kv is None else [b for _, b in kv],
                                         max_new=256 if kind == "step" else case["rows"] + 64)
        ids = torch.randint(0, case["vocab"], (max(case.get("rows", 1), 1),), device="cuda", generator=g).tolist()
        st["ids"] = ids
        if kind == "step":
            st["stage"].reset(ids[0])
            st["stage"].capture()
    else:
        raise ValueError(f"unknown kind {kind}")
    return st


# ---- one pass ----------------------------------------------------------------

def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "wire":
        header, payload = transport.encode(st["x"], case["codec"])
        return {"payload": payload, "x": transport.decode(header, payload)}
    if kind == "dropin":
        return st["op"](st["x"])
    if kind == "layer":
        st["graph"].replay()
        ctx = case["context"]
        return {"x": st["x2"], "mlp": st["mlp_out"], "k": st["k_cache"][:, ctx], "v": st["v_cache"][:, ctx]}
    if kind == "decode_attention":
        _decode_attention(case, st, st["q"], st["k"], st["v"])
        ctx = case["context"]
        return {"attn": st["attn"], "k": st["k_cache"][:, ctx], "v": st["v_cache"][:, ctx]}
    if kind == "mlp":
        q4.mlp_dev(st["gate"], st["up"], st["down"], st["x"], h=st["h"], out=st["out"])
        return {"h": st["h"], "out": st["out"]}
    if kind == "linear":
        return q4.gemv_multi_dev(st["mats"], st["x"], outs=st["outs"])
    if kind == "prompt_linear":
        return q4.gemm_bf16_multi_dev(st["mats"], st["x"], outs=st["outs"])
    if kind == "prompt_mlp":
        q4.gemm_bf16_gate_up_silu_dev(st["gate"], st["up"], st["x"], h=st["h"])
        q4.gemm_bf16_multi_dev([st["down"]], st["h"], outs=[st["out"]])
        return {"h": st["h"], "out": st["out"]}
    if kind == "prompt_attention":
        lib = st["lib"]
        fn = lib.q4_prompt_attention_bf16_dev if case["out_bf16"] else lib.q4_prompt_attention_dev
        q4.check(lib, fn(st["q"].data_ptr(), st["k_cache"].data_ptr(), st["v_cache"].data_ptr(),
                         st["out"].data_ptr(), case["rows"], case["context"], case["heads"], case["kv_heads"],
                         case["head_dim"], st["cap"], st["scale"], torch.cuda.current_stream().cuda_stream),
                 "prompt attention")
        return st["out"]
    if kind == "sweep":
        st["chain"].run()
        return st["out"]
    stage, ctx = st["stage"], case["context"]
    if kind == "step":
        stage.reset(st["ids"][0])
        tok = stage.step()
        rows = slice(ctx, ctx + 1)
    else:
        stage.truncate(ctx)
        tok = stage.prefill(st["ids"])
        rows = slice(ctx, ctx + case["rows"])
    return {"token": tok, "logits": stage.logits, "k": [L["k_cache"][:, rows] for L in stage.layers],
            "v": [L["v_cache"][:, rows] for L in stage.layers]}


# ---- what a pass cannot do without -------------------------------------------

def _w_bytes(n_out, n_in, gs=64):
    return n_out * n_in // 2 + 4 * n_out * (n_in // gs)


def _layer_work(h, inter, kvd):
    shapes = [(h, h), (kvd, h), (kvd, h), (h, h), (inter, h), (inter, h), (h, inter)]
    return sum(_w_bytes(n, k) for n, k in shapes), sum(2 * n * k for n, k in shapes)


def work(case):
    kind = case["kind"]
    if kind == "wire":
        n = case["rows"] * case["hidden"]
        payload = 2 * n if case["codec"] == "fp16" else n + 4 * case["rows"]
        return {"bytes": 8 * n + 2 * payload, "flops": 4 * n}
    if kind == "dropin":
        m, n, k = case["rows"], case["n_out"], case["n_in"]
        return {"bytes": _w_bytes(n, k, case["gs"]) + 4 * m * (n + k), "flops": 2 * m * n * k}
    if kind in ("layer", "decode_attention"):
        h, kv, d, n = case["heads"], case["kv_heads"], case["head_dim"], case["context"] + 1
        by, fl = 4 * kv * n * d + 8 * h * d, 4 * h * n * d
        if kind == "layer":
            wb, wf = _layer_work(case["hidden"], case["inter"], kv * d)
            by, fl = by + wb + 16 * case["hidden"], fl + wf
        return {"bytes": by, "flops": fl}
    if kind in ("mlp", "prompt_mlp"):
        m, h, i, gs = case["rows"], case["hidden"], case["inter"], case.get("gs", 64)
        act = 8 * m * h + 4 * m * i if kind == "mlp" else 6 * m * h + 2 * m * i
        return {"bytes": 2 * _w_bytes(i, h, gs) + _w_bytes(h, i, gs) + act, "flops": 6 * m * h * i}
    if kind in ("linear", "prompt_linear"):
        m, k, gs = case["rows"], case["n_in"], case.get("gs", 64)
        return {"bytes": sum(_w_bytes(n, k, gs) + 4 * m * n for n in _outs(case)) + (2 if case.get("x_bf16") else 4) * m * k,
                "flops": sum(2 * m * n * k for n in _outs(case))}
    if kind == "prompt_attention":
        r, c, h, kv, d = case["rows"], case["context"], case["heads"], case["kv_heads"], case["head_dim"]
        pairs = r * c + r * (r + 1) // 2
        return {"bytes": 4 * kv * (c + r) * d + (4 + (2 if case["out_bf16"] else 4)) * r * h * d, "flops": 4 * h * d * pairs}
    if kind == "sweep":
        layer, head = _sweep_shapes(case)
        shapes = [s for ph in layer for s in ph] * case["layers"] + [head]
        return {"bytes": sum(_w_bytes(n, k) + 4 * n for n, k in shapes) + 4 * (case["hidden"] + case["inter"]),
                "flops": sum(2 * n * k for n, k in shapes)}
    wb, wf = _layer_work(HIDDEN, INTER, KV_HEADS * HEAD_DIM)
    m, c, layers = case.get("rows", 1), case["context"], case["layers"]
    pairs = m * c + m * (m + 1) // 2
    return {"bytes": layers * (wb + 4 * KV_HEADS * (c + m) * HEAD_DIM) + _w_bytes(case["vocab"], HIDDEN) + 4 * case["vocab"],
            "flops": layers * (m * wf + 4 * HEADS * HEAD_DIM * pairs) + 2 * case["vocab"] * HIDDEN}


# ---- how far another correct implementation may be ---------------------------

def tolerance(case):
    kind = case["kind"]
    if kind in ("wire", "dropin", "linear", "sweep"):
        return "exact"               # the interface promises the reference arithmetic bit for bit
    # four times what the path was measured to move when its sums are taken in another order or its inputs by one
    # rounding of 32 bits.  A GEMV behind such a change quantises its x to 16-bit integers anew, which moves some
    # values by one step (mlp, layer); values stored in 16 bits (the cache, bf16 outputs) may move by one unit.
    if kind == "prompt_attention" and case["out_bf16"]:
        return {"rel": 1.7e-4, "max": 0.032}
    if kind == "prefill":            # bf16 operands: grows with each layer that a rounding travels through
        return {"rel": [7.3e-3, 0.026, 0.03][min(case["layers"], 3) - 1], "max": [0.033, 0.12, 0.2][min(case["layers"], 3) - 1]}
    return {"layer": {"rel": 1.2e-3, "max": 4e-3}, "decode_attention": {"rel": 1.5e-6, "max": 8e-6},
            "mlp": {"rel": 3.2e-4, "max": 1.6e-3}, "prompt_linear": {"rel": 1e-6, "max": 1e-5},
            "prompt_mlp": {"rel": 1.6e-4, "max": 0.032}, "prompt_attention": {"rel": 2e-6, "max": 1.4e-5},
            "step": {"rel": 1.3e-2, "max": 0.075}}[kind]


# ---- the same in 64 bits -----------------------------------------------------

def _deq(mat):
    w, s, b = mat
    sh = torch.arange(8, dtype=torch.int32, device=w.device) * 4
    q = ((w.unsqueeze(-1) >> sh) & 15).reshape(w.shape[0], s.shape[1], -1).double()
    v = q * s.view(torch.float16).double().unsqueeze(-1) + b.view(torch.float16).double().unsqueeze(-1)
    return v.reshape(w.shape[0], -1)


def _mm64(x, mat, block=8192):
    """x @ dequant(mat)^T in float64, a block of rows at a time."""
    w, s, b = mat
    return torch.cat([x @ _deq((w[i:i + block], s[i:i + block], b[i:i + block])).t().contiguous()
                      for i in range(0, w.shape[0], block)], dim=1)


def _silu_mul64(g, u):
    return g / (1 + torch.exp(-g)) * u


def _norm64(x, w, eps=1e-6):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w.double()


def _rope64(t, cos, sin):
    """t [rows, heads, d], cos and sin [rows, d/2]."""
    half = t.shape[-1] // 2
    a, b, c, s = t[..., :half], t[..., half:], cos.double().unsqueeze(1), sin.double().unsqueeze(1)
    return torch.cat([a * c - b * s, b * c + a * s], dim=-1)


def _attend64(q, k, v, scale, pos0):
    """q [rows, heads, d] at positions pos0.., k and v [kv_heads, positions, d]; causal."""
    rows, heads, d = q.shape
    group = heads // k.shape[0]
    n = pos0 + rows
    out = torch.empty((rows, heads, d), dtype=torch.float64, device=q.device)
    ahead = torch.arange(n, device=q.device)[None, :] > (torch.arange(rows, device=q.device) + pos0)[:, None]
    for h in range(heads):
        s = q[:, h] @ k[h // group, :n].double().t().contiguous() * scale
        out[:, h] = torch.softmax(s.masked_fill(ahead, -math.inf), dim=-1) @ v[h // group, :n].double()
    return out


def _layer64(x, delta, L, heads, kv_heads, d, cos, sin, scale, pos0, eps):
    """One decoder layer on rows x: (x + attention, mlp, new keys, new values); the cache holds fp16 values."""
    rows = x.shape[0]
    x = x if delta is None else x + delta
    hn = _norm64(x, L["in_w"], eps)
    bias = L["qkv_bias"].double().split([heads * d, kv_heads * d, kv_heads * d])
    q, k, v = ((_mm64(hn, m) + b).reshape(rows, -1, d) for m, b in zip(L["qkv"], bias))
    q, k = _rope64(q, cos[pos0:pos0 + rows], sin[pos0:pos0 + rows]), _rope64(k, cos[pos0:pos0 + rows], sin[pos0:pos0 + rows])
    kn, vn = k.transpose(0, 1), v.transpose(0, 1)
    keys = torch.cat([L["k_cache"][:, :pos0].double(), kn.half().double()], dim=1)
    vals = torch.cat([L["v_cache"][:, :pos0].double(), vn.half().double()], dim=1)
    x = x + _mm64(_attend64(q, keys, vals, scale, pos0).reshape(rows, -1), L["o"])
    hn = _norm64(x, L["post_w"], eps)
    return x, _mm64(_silu_mul64(_mm64(hn, L["gate"]), _mm64(hn, L["up"])), L["down"]), kn, vn


def exact(case, seed):
    kind = case["kind"]
    st = prepare(case, seed)
    if kind == "wire":
        # the payload is bytes and the decoded values follow from their roundings
        return {"payload": None, "x": st["x"].double()}
    if kind == "dropin":
        op = st["op"]
        mat = tuple(torch.from_numpy(a).cuda() for a in (op.w.view(np.int32), op.scales.view(np.int16), op.biases.view(np.int16)))
        return _mm64(torch.from_numpy(st["x"]).cuda().double(), mat).cpu().numpy()
    if kind == "layer":
        L = {"qkv": st["qkv"], "qkv_bias": st["bias"], "o": st["o"], "gate": st["gate"], "up": st["up"],
             "down": st["down"], "in_w": st["in_w"], "post_w": st["post_w"], "k_cache": st["k_cache"],
             "v_cache": st["v_cache"]}
        x, mlp, k, v = _layer64(st["x"].double()[None], st["delta"].double()[None], L, case["heads"], case["kv_heads"],
                                case["head_dim"], st["cos"], st["sin"], st["scale"], case["context"], 1e-6)
        return {"x": x, "mlp": mlp, "k": k[:, 0], "v": v[:, 0]}
    if kind == "decode_attention":
        h, kv, d, pos = case["heads"], case["kv_heads"], case["head_dim"], case["context"]
        q, k, v = ((st[n].double() + b.double()).reshape(1, -1, d)
                   for n, b in zip("qkv", st["bias"].split([h * d, kv * d, kv * d])))
        cos, sin = st["cos"][pos:pos + 1], st["sin"][pos:pos + 1]
        q, k = _rope64(q, cos, sin), _rope64(k, cos, sin)
        keys = torch.cat([st["k_cache"][:, :pos].double(), k.transpose(0, 1).half().double()], dim=1)
        vals = torch.cat([st["v_cache"][:, :pos].double(), v.transpose(0, 1).half().double()], dim=1)
        return {"attn": _attend64(q, keys, vals, st["scale"], pos).reshape(1, -1), "k": k[0], "v": v[0]}
    if kind in ("mlp", "prompt_mlp"):
        x = st["x"].double()
        h = _silu_mul64(_mm64(x, st["gate"]), _mm64(x, st["up"]))
        return {"h": h, "out": _mm64(h, st["down"])}
    if kind in ("linear", "prompt_linear"):
        return [_mm64(st["x"].double(), m) for m in st["mats"]]
    if kind == "prompt_attention":
        d = case["head_dim"]
        out = _attend64(st["q"].double().reshape(case["rows"], -1, d), st["k_cache"], st["v_cache"], st["scale"], case["context"])
        return out.reshape(case["rows"], -1)
    if kind == "sweep":
        out = torch.zeros(st["out"].shape, dtype=torch.float64, device="cuda")
        for mats, x, outs, _ in st["phases"]:
            for m, o in zip(mats, outs):
                out[o.storage_offset():o.storage_offset() + o.numel()] = _mm64(x.double(), m)[0]
        return out
    stage = st["stage"]
    ids = torch.tensor(st["ids"], device="cuda")
    x = _deq(tuple(t[ids] for t in stage.embed))
    delta, ks, vs = None, [], []
    for L in stage.layers:
        x, delta, k, v = _layer64(x, delta, L, HEADS, KV_HEADS, HEAD_DIM, stage.cos, stage.sin, stage.scale,
                                  case["context"], stage.eps)
        ks.append(k)
        vs.append(v)
    logits = _mm64(_norm64(x[-1:] + delta[-1:], stage.norm_w, stage.eps), stage.lm_head)
    return {"token": None, "logits": logits, "k": ks, "v": vs}
