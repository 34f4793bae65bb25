"""The framework's work as its users call it: the cases that its speed is measured on.

Three kinds of program use the library: one that holds the qkv projections and calls the
window attention (AWA) op layer by layer, in bf16 or fp32 storage; one that runs whole DiT
layers on a residual stream; and one that runs the whole DiT, from the latent grid to the
latent output.  The cases cover each of them over the latent grids of the repository's tests
and bench (360p, 720p, 1080p, the ragged 71x97 grid, several frames) with both window
geometries.  `listed` names the fixed cases, `draw` gives others of the same ranges.

All inputs come from the seed alone and are made on the GPU.  Activations and q, k, v are
N(0, 1), linear weights N(0, 0.02), qk-norm gains and modulation scales 1 + N(0, 0.02), the
other modulation vectors N(0, 0.02), the branch gates N(0, 0.5).
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "seedvr2-2b-ncnn_amd"))

import awa_hip  # noqa: E402

HEADS, HEAD_D, DIM, QKV = 20, 128, 2560, 7680
MLP = 6912            # the checkpoint's SwiGLU width
EPS = 1e-5
DUAL_LAYERS = 10      # of a whole model's layers, those with separate text weights
ADA = ("attn_shift", "attn_scale", "attn_gate", "mlp_shift", "mlp_scale", "mlp_gate")


# ------------------------------------------------------------------ the cases

def _awa(name, grid, nw, txt, shifted, dtype, outliers=0.0):
    return {"name": name, "kind": "awa", "t": grid[0], "h": grid[1], "w": grid[2], "nt": nw[0], "nh": nw[1],
            "nw": nw[2], "txt": txt, "shifted": shifted, "dtype": dtype, "outliers": outliers}


def _dit(name, kind, grid, txt, shifted=False, dual=False, layers=1):
    """A case of the DiT around the op; (t, h, w) is the token grid, half the latent grid."""
    return {"name": name, "kind": kind, "t": grid[0], "h": grid[1], "w": grid[2], "nt": 4, "nh": 3, "nw": 3,
            "txt": txt, "shifted": shifted, "dual": dual, "layers": layers}


def listed():
    return [
        # the smallest call: a thumbnail's grid with a short prompt, bounded by launches
        _awa("awa_tiny_bf16", (1, 12, 20), (4, 3, 3), 9, False, "bf16"),
        # a program that keeps the reference's fp32 storage: 360p, and the same at 1080p
        _awa("awa_360p_f32", (1, 23, 27), (4, 3, 3), 58, False, "f32"),
        _awa("awa_1080p_f32_shifted", (1, 68, 80), (4, 3, 3), 58, True, "f32"),
        # the op of a bf16 model's layers: an odd layer at 720p, an even one at 1080p
        _awa("awa_720p_bf16_shifted", (1, 45, 53), (4, 3, 3), 58, True, "bf16"),
        _awa("awa_1080p_bf16", (1, 68, 80), (4, 3, 3), 58, False, "bf16"),
        # a grid that no window size divides, a longer prompt, activations with outliers
        _awa("awa_ragged_bf16_shifted", (1, 71, 97), (1, 4, 4), 77, True, "bf16", 0.01),
        # a clip: five latent frames of 1080p
        _awa("awa_video_bf16_shifted", (5, 68, 80), (4, 3, 3), 58, True, "bf16"),
        # one DiT layer: an early one (separate text weights) at 360p, a later one at 1080p
        _dit("layer_360p_dual", "layer", (1, 23, 27), 58, False, True),
        _dit("layer_1080p_shifted", "layer", (1, 68, 80), 58, True, False),
        # the model's two ends at 1080p: latent grid and prompt to the residual stream, and back
        _dit("embed_1080p", "embed", (1, 68, 80), 58),
        _dit("final_1080p", "final", (1, 68, 80), 58),
        # the whole denoising step at 1080p: 32 layers, latent grid in, latent grid out
        _dit("step_1080p", "step", (1, 68, 80), 58, False, True, 32),
    ]


def _grid(rng, lo, hi, frames):
    """A token grid of lo..hi rows (log-uniform), 1 to `frames` frames, aspect 1:3 to 3:1."""
    while True:
        rows = math.exp(rng.uniform(math.log(lo), math.log(hi)))
        t = rng.randint(1, frames)
        aspect = math.exp(rng.uniform(-math.log(3), math.log(3)))
        h = max(1, round(math.sqrt(rows / t * aspect)))
        w = max(1, round(rows / t / h))
        if lo <= t * h * w <= hi:
            return t, h, w


def draw(rng):
    kind = rng.choice(["awa", "awa", "awa", "awa", "layer", "layer", "embed", "final", "step"])
    txt = rng.randint(1, 140)
    shifted = rng.random() < 0.5
    if kind == "awa":
        f32 = rng.random() < 0.3
        c = _awa("", _grid(rng, 200, 6000 if f32 else 27200, 5), rng.choice([(4, 3, 3), (4, 3, 3), (1, 4, 4), (2, 2, 3)]),
                 txt, shifted, "f32" if f32 else "bf16", rng.choice([0.0, 0.0, 0.01]))
    elif kind == "step":
        c = _dit("", kind, _grid(rng, 200, 5000, 3), txt, False, True, rng.randint(2, 32))
    elif kind == "layer":
        c = _dit("", kind, _grid(rng, 200, 12000, 3), txt, shifted, rng.random() < 0.4)
    else:
        c = _dit("", kind, _grid(rng, 200, 12000, 3), txt)
    del c["name"]
    return c


# ------------------------------------------------------------------ inputs

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _randn(g, *shape, scale=1.0, mean=0.0, dtype=torch.float32):
    x = torch.randn(shape, generator=g, device="cuda", dtype=torch.float32)
    if scale != 1.0:
        x *= scale
    if mean != 0.0:
        x += mean
    return x.to(dtype)


def _rows(c):
    return c["t"] * c["h"] * c["w"]


def _awa_inputs(c, seed):
    g = _gen(seed)
    dt = torch.float32 if c["dtype"] == "f32" else torch.bfloat16
    out = []
    for n in (_rows(c), c["txt"]):
        x = _randn(g, n, QKV)
        if c["outliers"] > 0:
            x = torch.where(torch.rand(x.shape, generator=g, device="cuda") < c["outliers"], 8 * x, x)
        out.append(x.to(dt))
    return out[0], out[1], [_randn(g, HEAD_D, scale=0.02, mean=1.0) for _ in range(4)]


def _branch(g):
    bf = torch.bfloat16
    b = {"qkv_w": _randn(g, QKV, DIM, scale=0.02, dtype=bf), "out_w": _randn(g, DIM, DIM, scale=0.02, dtype=bf),
         "out_b": _randn(g, DIM, scale=0.02), "mlp_in_w": _randn(g, MLP, DIM, scale=0.02, dtype=bf),
         "mlp_g_w": _randn(g, MLP, DIM, scale=0.02, dtype=bf), "mlp_out_w": _randn(g, DIM, MLP, scale=0.02, dtype=bf),
         "nq": _randn(g, HEAD_D, scale=0.02, mean=1.0), "nk": _randn(g, HEAD_D, scale=0.02, mean=1.0)}
    for k in ADA:
        b[k] = _randn(g, DIM, scale=0.5 if "gate" in k else 0.02, mean=1.0 if "scale" in k else 0.0)
    return b


def _io(g):
    bf = torch.bfloat16
    return {"vid_in_w": _randn(g, DIM, 132, scale=0.02, dtype=bf), "vid_in_b": _randn(g, DIM, scale=0.02),
            "txt_in_w": _randn(g, DIM, 5120, scale=0.02, dtype=bf), "txt_in_b": _randn(g, DIM, scale=0.02),
            "out_norm_w": _randn(g, DIM, scale=0.02, mean=1.0), "out_ada_shift": _randn(g, DIM, scale=0.02),
            "out_ada_scale": _randn(g, DIM, scale=0.02, mean=1.0), "vid_out_w": _randn(g, 64, DIM, scale=0.02, dtype=bf),
            "vid_out_b": _randn(g, 64, scale=0.02)}


def _time_weights(g):
    return [_randn(g, *s, scale=0.02) for s in ((DIM, 256), (DIM,), (DIM, DIM), (DIM,), (6 * DIM, DIM), (6 * DIM,))]


def _dit_inputs(c, seed):
    """Everything of a DiT case as plain tensors; the branches' MLP weights unpacked."""
    g = _gen(seed)
    d = {}
    if c["kind"] in ("layer", "final"):
        d["x"] = _randn(g, _rows(c) + c["txt"], DIM)
        d["emb"] = _randn(g, 6 * DIM, scale=0.02)
    if c["kind"] in ("embed", "step"):
        d["grid"] = _randn(g, c["t"], 2 * c["h"], 2 * c["w"], 33)
        d["text"] = _randn(g, c["txt"], 5120)
    if c["kind"] != "layer":
        d["io"] = _io(g)
    if c["kind"] == "step":
        d["time"] = _time_weights(g)
    if c["kind"] in ("layer", "step"):
        dual = DUAL_LAYERS if c["kind"] == "step" else int(c["dual"])
        d["branches"] = []
        for i in range(c["layers"]):
            vid = _branch(g)
            d["branches"].append((vid, _branch(g) if i < dual else vid))
    return d


def _packed(ctx, b):
    """A branch as the library takes it, the SwiGLU weights interleaved once."""
    p = {k: v for k, v in b.items() if k not in ("mlp_in_w", "mlp_g_w")}
    p["mlp_w"] = ctx.pack_mlp(b["mlp_in_w"], b["mlp_g_w"])
    return p


def prepare(case, seed):
    c = case
    ctx = awa_hip.Context(0)
    windows = (c["nt"], c["nh"], c["nw"])

    def geometry(shifted):
        return ctx.build_geometry(c["t"], c["h"], c["w"], windows, c["txt"], shifted)

    s = {"case": c, "ctx": ctx}
    if c["kind"] == "awa":
        s["vqkv"], s["tqkv"], s["gains"] = _awa_inputs(c, seed)
        s["geom"] = geometry(c["shifted"])
        ctx.reserve(s["geom"], c["dtype"])
        s["vattn"] = torch.empty((_rows(c), DIM), dtype=s["vqkv"].dtype, device="cuda")
        s["tattn"] = torch.empty((c["txt"], DIM), dtype=s["vqkv"].dtype, device="cuda")
        return s
    d = _dit_inputs(c, seed)
    M = _rows(c) + c["txt"]
    s["even"] = geometry(c["shifted"])
    ctx.dit_reserve(s["even"], MLP)
    if c["kind"] == "step":
        s["odd"] = geometry(True)
        ctx.dit_reserve(s["odd"], MLP)
        s["time"] = d["time"]
    if "io" in d:
        s["io"] = ctx.io_layers(d["io"])
    if "branches" in d:
        s["layers"] = []
        for vid, txt in d["branches"]:
            pv = _packed(ctx, vid)
            s["layers"].append((pv, pv if txt is vid else _packed(ctx, txt)))
    for k in ("x", "emb", "grid", "text"):
        if k in d:
            s[k] = d[k]
    if c["kind"] != "final":
        s["stream"] = torch.empty((M, DIM), dtype=torch.float32, device="cuda")  # the residual stream
    if c["kind"] in ("final", "step"):
        s["out"] = torch.empty((c["t"], 2 * c["h"], 2 * c["w"], 16), dtype=torch.float32, device="cuda")
    return s


# ------------------------------------------------------------------ one pass

def run(state):
    s, c, ctx = state, state["case"], state["ctx"]
    if c["kind"] == "awa":
        return ctx.forward(s["geom"], s["vqkv"], s["tqkv"], *s["gains"], eps=EPS, vattn=s["vattn"], tattn=s["tattn"])
    if c["kind"] == "layer":
        # a layer works in place; the caller's hidden state stays as it is
        s["stream"].copy_(s["x"])
        vid, txt = s["layers"][0]
        return ctx.layer(s["even"], vid, txt, s["emb"], s["stream"], _rows(c), c["txt"], mlp=MLP, eps=EPS)
    if c["kind"] == "embed":
        return ctx.embed(s["io"], s["grid"], s["text"], x=s["stream"])
    if c["kind"] == "final":
        return ctx.final(s["io"], s["emb"], s["x"], c["t"], 2 * c["h"], 2 * c["w"], eps=EPS, out=s["out"])
    out = ctx.forward_grid(s["io"], s["time"], s["layers"], s["even"], s["odd"], 1000.0, s["grid"], s["text"], mlp=MLP,
                           eps=EPS, x=s["stream"], out=s["out"])
    return out, s["stream"]


# ------------------------------------------------------------------ the work of a pass

def _axis(X, size, shifted):
    """Slices of one axis (awa_window.cpp:15-78)."""
    out = []
    if not shifted:
        for i in range((X + size - 1) // size):
            out.append((i * size, min((i + 1) * size, X)))
    elif size >= X:
        out.append((0, X))
    else:
        for i in range(math.ceil((X - 0.5) / size) + 1):
            out.append((max(int((i - 0.5) * size), 0), min(int((i + 0.5) * size), X)))
    return [(a, b) for a, b in out if b > a]


def _windows(c, shifted):
    """[((t0, t1), (h0, h1), (w0, w1))] in the op's window order."""
    scale = math.sqrt(45 * 80 / (c["h"] * c["w"]))
    size = (math.ceil(min(c["t"], 30) / c["nt"]), math.ceil(math.floor(c["h"] * scale + 0.5) / c["nh"]),
            math.ceil(math.floor(c["w"] * scale + 0.5) / c["nw"]))
    ax = [_axis(X, n, shifted) for X, n in zip((c["t"], c["h"], c["w"]), size)]
    return [(t, h, w) for w in ax[2] for h in ax[1] for t in ax[0]]


def _awa_flops(c, shifted):
    total = 0
    for t, h, w in _windows(c, shifted):
        S = (t[1] - t[0]) * (h[1] - h[0]) * (w[1] - w[0]) + c["txt"]
        total += 4 * HEAD_D * HEADS * S * S
    return total


BRANCH_BYTES = 2 * (QKV * DIM + DIM * DIM + 3 * MLP * DIM) + 4 * (7 * DIM + 2 * HEAD_D)
TIME_BYTES = 4 * (DIM * 256 + DIM + DIM * DIM + DIM + 6 * DIM * DIM + 6 * DIM)


def work(case):
    c = case
    Lv, txt = _rows(c), c["txt"]
    M = Lv + txt
    if c["kind"] == "awa":
        elem = 4 if c["dtype"] == "f32" else 2
        return {"bytes": elem * M * (QKV + DIM) + 4 * 4 * HEAD_D, "flops": _awa_flops(c, c["shifted"])}
    stream = 4 * M * DIM
    gemms = 2 * M * DIM * (QKV + DIM + 3 * MLP)  # of a layer
    embed = {"bytes": 4 * (4 * Lv * 33 + txt * 5120) + 2 * DIM * (132 + 5120) + 2 * 4 * DIM,
             "flops": 2 * DIM * (Lv * 132 + txt * 5120)}
    final = {"bytes": 2 * 64 * DIM + 4 * (3 * DIM + 64 + 2 * DIM) + 4 * 4 * Lv * 16, "flops": 2 * Lv * DIM * 64}
    if c["kind"] == "embed":
        return {"bytes": embed["bytes"] + stream, "flops": embed["flops"]}
    if c["kind"] == "final":
        return {"bytes": final["bytes"] + 4 * Lv * DIM, "flops": final["flops"]}
    if c["kind"] == "layer":
        return {"bytes": (2 if c["dual"] else 1) * BRANCH_BYTES + 4 * 6 * DIM + 2 * stream,
                "flops": gemms + _awa_flops(c, c["shifted"])}
    n = c["layers"]
    return {"bytes": embed["bytes"] + final["bytes"] + TIME_BYTES + (n + min(n, DUAL_LAYERS)) * BRANCH_BYTES + stream,
            "flops": embed["flops"] + final["flops"] + n * gemms +
            sum(_awa_flops(c, i % 2 == 1) for i in range(n))}


def tolerance(case):
    """About four times the error against `exact` of outputs of the stated types."""
    c = case
    if c["kind"] == "awa":
        # fp32 storage: fp32 sums in another order
        if c["dtype"] == "f32":
            return {"rel": 4e-6}
        # bf16: q, k and probabilities as bf16 matrix operands, bf16 outputs (outliers sharpen the softmax)
        return {"rel": 2.4e-2 if c["outliers"] > 0 else 1.4e-2}
    # fp32 outputs of bf16 matrix operands; the step's 32 layers each feed the next
    return {"rel": {"layer": 6e-3, "embed": 7e-3, "final": 7e-3, "step": 7e-2}[c["kind"]]}


# ------------------------------------------------------------------ the same in 64 bits

def _f64(x):
    return x.to(torch.float64)


def _angles(pos, n):
    """[len(pos)][n] angles of one axis: float32(position / 10000^(2j/42)), as the windows' tables hold them."""
    base = torch.tensor([1.0 / math.pow(10000.0, 2 * j / 42) for j in range(n)], dtype=torch.float64, device="cuda")
    return _f64((_f64(pos)[:, None] * base[None, :]).to(torch.float32))


def _norm_rope(x, gain, ang):
    """Per-head RMSNorm with gain, then rotation of channel pairs 0..62: x [S, 20, 128], ang [S, 63]."""
    x = x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * _f64(gain)
    c, s = torch.cos(ang)[:, None, :], torch.sin(ang)[:, None, :]
    y = x.clone()
    a, b = x[..., 0:126:2], x[..., 1:126:2]
    y[..., 0:126:2] = a * c - b * s
    y[..., 1:126:2] = b * c + a * s
    return y


def _exact_awa(c, shifted, vqkv, tqkv, gains):
    """vqkv [Lv, 7680] and tqkv [txt, 7680] in 64 bits; gains of q and k, video then text."""
    txt, dev = c["txt"], "cuda"
    nq_v, nk_v, nq_t, nk_t = gains
    ti = _angles(torch.arange(txt, device=dev), 21)
    tang = torch.cat([ti, ti, ti], 1)
    tq, tk, tv = (tqkv[:, i * DIM:(i + 1) * DIM].reshape(txt, HEADS, HEAD_D) for i in range(3))
    tq, tk = _norm_rope(tq, nq_t, tang), _norm_rope(tk, nk_t, tang)
    vout = torch.zeros((_rows(c), DIM), dtype=torch.float64, device=dev)
    tout = torch.zeros((txt, DIM), dtype=torch.float64, device=dev)
    wins = _windows(c, shifted)
    for t, h, w in wins:
        n = [b - a for a, b in (t, h, w)]
        it, ih, iw = (v.reshape(-1) for v in torch.meshgrid(*[torch.arange(k, device=dev) for k in n], indexing="ij"))
        idx = ((t[0] + it) * c["h"] + h[0] + ih) * c["w"] + w[0] + iw
        ang = torch.cat([_angles(txt + it, 21), _angles(ih, 21), _angles(iw, 21)], 1)
        rows = vqkv[idx]
        q, k, v = (rows[:, i * DIM:(i + 1) * DIM].reshape(-1, HEADS, HEAD_D) for i in range(3))
        q = torch.cat([_norm_rope(q, nq_v, ang), tq]).transpose(0, 1)
        k = torch.cat([_norm_rope(k, nk_v, ang), tk]).transpose(0, 1)
        v = torch.cat([v, tv]).transpose(0, 1)
        p = torch.softmax(q @ k.transpose(1, 2).contiguous() / math.sqrt(HEAD_D), -1)
        o = (p @ v.contiguous()).transpose(0, 1).reshape(-1, DIM)
        vout[idx] = o[:idx.numel()]
        tout += o[idx.numel():]
    return vout, tout / len(wins)


def _rms(x):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS)


def _exact_layer(c, shifted, x, emb, vid, txt):
    Lv, outs = _rows(c), []
    e = _f64(emb)
    mod = [{k: e[j::6] + _f64(b[k]) for j, k in enumerate(ADA)} for b in (vid, txt)]
    halves = [x[:Lv], x[Lv:]]
    qkv = [(_rms(p) * m["attn_scale"] + m["attn_shift"]) @ _f64(b["qkv_w"]).T
           for p, m, b in zip(halves, mod, (vid, txt))]
    att = _exact_awa(c, shifted, qkv[0], qkv[1], (vid["nq"], vid["nk"], txt["nq"], txt["nk"]))
    for p, a, m, b in zip(halves, att, mod, (vid, txt)):
        y = p + m["attn_gate"] * (a @ _f64(b["out_w"]).T + _f64(b["out_b"]))
        h = _rms(y) * m["mlp_scale"] + m["mlp_shift"]
        g = h @ _f64(b["mlp_g_w"]).T
        u = g * torch.sigmoid(g) * (h @ _f64(b["mlp_in_w"]).T)
        outs.append(y + m["mlp_gate"] * (u @ _f64(b["mlp_out_w"]).T))
    return torch.cat(outs)


def _exact_embed(c, io, grid, text):
    t, h, w = c["t"], c["h"], c["w"]
    p = _f64(grid).reshape(t, h, 2, w, 2, 33).permute(0, 1, 3, 2, 4, 5).reshape(-1, 132)
    return torch.cat([p @ _f64(io["vid_in_w"]).T + _f64(io["vid_in_b"]),
                      _f64(text) @ _f64(io["txt_in_w"]).T + _f64(io["txt_in_b"])])


def _exact_final(c, io, emb, x):
    t, h, w = c["t"], c["h"], c["w"]
    e = _f64(emb)
    y = _rms(x[:_rows(c)]) * _f64(io["out_norm_w"])
    y = y * (e[1::6] + _f64(io["out_ada_scale"])) + e[0::6] + _f64(io["out_ada_shift"])
    y = y @ _f64(io["vid_out_w"]).T + _f64(io["vid_out_b"])
    return y.reshape(t, h, w, 2, 2, 16).permute(0, 1, 3, 2, 4, 5).reshape(t, 2 * h, 2 * w, 16).contiguous()


def _exact_time(t, tw):
    w_in, b_in, w_hid, b_hid, w_out, b_out = (_f64(w) for w in tw)
    f = torch.tensor([math.exp(-math.log(10000.0) * j / 128) for j in range(128)], dtype=torch.float64, device="cuda")
    y = torch.cat([torch.sin(t * f), torch.cos(t * f)])
    y = torch.nn.functional.silu(w_in @ y + b_in)
    y = torch.nn.functional.silu(w_hid @ y + b_hid)
    return w_out @ y + b_out


def exact(case, seed):
    c = case
    if c["kind"] == "awa":
        vqkv, tqkv, gains = _awa_inputs(c, seed)
        return _exact_awa(c, c["shifted"], _f64(vqkv), _f64(tqkv), gains)
    d = _dit_inputs(c, seed)
    if c["kind"] == "layer":
        return _exact_layer(c, c["shifted"], _f64(d["x"]), d["emb"], *d["branches"][0])
    if c["kind"] == "final":
        return _exact_final(c, d["io"], d["emb"], _f64(d["x"]))
    x = _exact_embed(c, d["io"], d["grid"], d["text"])
    if c["kind"] == "embed":
        return x
    emb = _exact_time(1000.0, d["time"])
    for i, (vid, txt) in enumerate(d["branches"]):
        x = _exact_layer(c, i % 2 == 1, x, emb, vid, txt)
    return _exact_final(c, d["io"], emb, x), x
