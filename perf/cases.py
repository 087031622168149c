"""What a program built on this framework spends its time on, as measurable cases.

A robot runs whole chunks (``SmolVLAEngine``: one sample for latency, a batch
for throughput).  A program with its own composition calls the layers, each
through the function a reference caller binds (``smolvla.vla``): the vision
block, the decoder (prefix) layer, the expert's self and cross layers, the
connector, the patch embedding.  Sizes are the model's own -- 1024 ViT tokens
of 768, a prefix of up to 241 rows of 960, 50 action rows of 720, three
cameras, batches from 1 to 32 -- and, since every layer takes any length, odd
and ragged ones.


A layer is called either eagerly (``via="call"``) or, as latency-minded
programs and the engine itself do, captured once into a HIP graph and replayed
on fresh inputs (``via="graph"``).

``exact`` restates each path in plain float64 torch.
"""

import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "vla-to-npu_amd"))

BF16 = torch.bfloat16
F32 = torch.float32
F64 = torch.float64

VIT = dict(hidden=768, heads=12, inter=3072, layers=12, image=512, patch=16, chans=3)
DEC = dict(hidden=960, q=15, kv=5, inter=2560, layers=16)
EXP = dict(hidden=720, q=15, kv=5, inter=2048, layers=16)
HD = 64
THETA, RMS_EPS, LN_EPS = 100000.0, 1e-5, 1e-6
VOCAB, STATE, ACTION, CHUNK, STEPS, SHUFFLE = 49152, 32, 32, 50, 10, 4


# ------------------------------------------------------------------ cases ---
def listed():
    return [
        # the control loop of one robot: one sample, latency is all that counts
        dict(name="chunk_1", kind="chunk", batch=1, cameras=3, lang=48),
        # a server that batches requests: the framework's throughput figure
        dict(name="chunk_32", kind="chunk", batch=32, cameras=3, lang=48),
        # one camera frame through a vision block
        dict(name="vit_1x1024", kind="vit", images=1, tokens=1024, gelu="tanh", biases=True,
             via="graph"),
        # 32 samples of 3 cameras through a vision block
        dict(name="vit_96x1024", kind="vit", images=96, tokens=1024, gelu="tanh", biases=True,
             via="call"),
        # 384-pixel frames in 14-pixel patches (27 x 27 tokens: no tile divides
        # them), the reference module's own erf GELU, no projection biases
        dict(name="vit_7x729", kind="vit", images=7, tokens=729, gelu="erf", biases=False,
             via="graph"),
        # one prompt through a decoder layer: the smallest ordinary call
        dict(name="text_1x128", kind="text", batch=1, length=128, mask="causal", via="call"),
        # the prefix of a batch of 32
        dict(name="text_32x241", kind="text", batch=32, length=241, mask="prefix_lm",
             via="graph"),
        # a handful of longer, odd prompts
        dict(name="text_5x333", kind="text", batch=5, length=333, mask="causal", via="graph"),
        # one Euler step's self layer at batch 32
        dict(name="self_32x50", kind="self", batch=32, length=50, via="graph"),
        # one robot's cross layer on its prefix
        dict(name="cross_1x50x241", kind="cross", batch=1, length=50, context=241,
             via="graph"),
        # one observation's three cameras into the prefix
        dict(name="connector_3", kind="connector", images=3, via="call"),
        # a batch of 32 observations into the vision encoder
        dict(name="patch_96", kind="patch", images=96, via="call"),
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["chunk", "vit", "vit", "text", "text", "self", "cross", "connector",
                       "patch"])
    if kind == "chunk":
        return dict(kind=kind, batch=_log(rng, 1, 32), cameras=rng.randint(1, 3),
                    lang=rng.randint(8, 48))
    via = rng.choice(["graph", "graph", "call"])
    if kind == "vit":
        # frames of 14 to 32 patches a side
        return dict(kind=kind, images=_log(rng, 1, 96), tokens=rng.randint(14, 32) ** 2,
                    gelu=rng.choice(["tanh", "tanh", "erf"]), biases=rng.random() < 0.7, via=via)
    if kind == "text":
        mask = rng.choice(["causal", "prefix_lm"])
        return dict(kind=kind, batch=_log(rng, 1, 32), length=_log(rng, 17, 512), mask=mask,
                    via=via)
    if kind == "self":
        return dict(kind=kind, batch=_log(rng, 1, 64), length=rng.randint(10, 64), via=via)
    if kind == "cross":
        return dict(kind=kind, batch=_log(rng, 1, 64), length=rng.randint(10, 64),
                    context=rng.randint(65, 320), via=via)
    return dict(kind=kind, images=_log(rng, 1, 96), via=via)


# ----------------------------------------------------------------- inputs ---
class _Gen:
    """Weights N(0, 0.02), gains around 1, activations N(0, 1), pixels U(-1, 1)."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(seed)

    def normal(self, *shape, std=1.0, dtype=BF16):
        t = torch.randn(*shape, generator=self.g, device="cuda", dtype=F32)
        return (t * std).to(dtype)

    def lin(self, *shape):
        return self.normal(*shape, std=0.02)

    def gain(self, n):
        return (1.0 + self.normal(n, std=0.1, dtype=F32)).to(BF16)

    def pixels(self, *shape):
        t = torch.rand(*shape, generator=self.g, device="cuda", dtype=F32)
        return (t * 2 - 1).to(BF16)

    def ids(self, *shape):
        return torch.randint(0, VOCAB, shape, generator=self.g, device="cuda")


def _decoder_params(g, c):
    H, q, kv, inter = c["hidden"], c["q"] * HD, c["kv"] * HD, c["inter"]
    return dict(Wq=g.lin(H, q), Wk=g.lin(H, kv), Wv=g.lin(H, kv), Wo=g.lin(q, H),
                W_gate=g.lin(H, inter), W_up=g.lin(H, inter), W_down=g.lin(inter, H),
                W_norm_1=g.gain(H), W_norm_2=g.gain(H))


def _cross_params(g, c, kv_in):
    p = _decoder_params(g, c)
    del p["Wk"], p["Wv"]
    p.update(Wk_cross=g.lin(kv_in, c["kv"] * HD), Wv_cross=g.lin(kv_in, c["kv"] * HD))
    return p


def _vit_params(g, biases):
    H, inter = VIT["hidden"], VIT["inter"]
    p = dict(Wq=g.lin(H, H), Wk=g.lin(H, H), Wv=g.lin(H, H), Wo=g.lin(H, H),
             W_up=g.lin(H, inter), W_down=g.lin(inter, H), W_norm_1=g.gain(H),
             b_norm_1=g.normal(H, std=0.1), W_norm_2=g.gain(H), b_norm_2=g.normal(H, std=0.1))
    if biases:
        p.update(bq=g.lin(H), bk=g.lin(H), bv=g.lin(H), bo=g.lin(H), b_up=g.lin(inter),
                 b_down=g.lin(H))
    return p


def _patch_params(g):
    E = VIT["hidden"]
    return dict(kernel=g.lin(E, VIT["chans"], VIT["patch"], VIT["patch"]), bias=g.lin(E),
                pos_emb=g.lin((VIT["image"] // VIT["patch"]) ** 2, E))


def _chunk_params(g):
    H = EXP["hidden"]
    kv = DEC["kv"] * HD
    return dict(
        patch=_patch_params(g), vit=[_vit_params(g, True) for _ in range(VIT["layers"])],
        connector=dict(W=g.lin(VIT["hidden"] * SHUFFLE ** 2, DEC["hidden"])),
        embed=g.lin(VOCAB, DEC["hidden"]), state=dict(W=g.lin(STATE, DEC["hidden"])),
        prefix=[_decoder_params(g, DEC) for _ in range(DEC["layers"])],
        expert=[_cross_params(g, EXP, kv) if i % 2 else _decoder_params(g, EXP)
                for i in range(EXP["layers"])],
        expert_io=dict(W_action_in=g.lin(ACTION, H), b_action_in=g.lin(H),
                       W_time_in=g.lin(2 * H, H), b_time_in=g.lin(H), W_time_out=g.lin(H, H),
                       b_time_out=g.lin(H), W_exp_norm=g.gain(H), W_action_out=g.lin(H, ACTION)))


def _inputs(case, seed):
    """(weights, inputs) of a case, made from the seed alone."""
    g = _Gen(seed)
    kind = case["kind"]
    if kind == "chunk":
        B, S = case["batch"], VIT["image"]
        return _chunk_params(g), (g.pixels(B, case["cameras"], VIT["chans"], S, S),
                                  g.ids(B, case["lang"]), g.normal(B, STATE, dtype=F32),
                                  g.normal(B, CHUNK, ACTION, dtype=F32))
    if kind == "vit":
        return _vit_params(g, case["biases"]), (
            g.normal(case["images"], case["tokens"], VIT["hidden"]),)
    if kind == "text":
        return _decoder_params(g, DEC), (g.normal(case["batch"], case["length"], DEC["hidden"]),)
    if kind == "self":
        return _decoder_params(g, EXP), (g.normal(case["batch"], case["length"], EXP["hidden"]),)
    if kind == "cross":
        kv = DEC["kv"] * HD
        return _cross_params(g, EXP, kv), (
            g.normal(case["batch"], case["length"], EXP["hidden"]),
            g.normal(case["batch"], case["context"], kv),
            g.normal(case["batch"], case["context"], kv))
    if kind == "connector":
        return dict(W=g.lin(VIT["hidden"] * SHUFFLE ** 2, DEC["hidden"])), (
            g.normal(case["images"], 1024, VIT["hidden"]),)
    if kind == "patch":
        return _patch_params(g), (
            g.pixels(case["images"], VIT["chans"], VIT["image"], VIT["image"]),)
    raise ValueError(kind)


def _chunk_config(case):
    from smolvla.config import SmolVLAConfig
    return SmolVLAConfig(n_cameras=case["cameras"], lang_tokens=case["lang"])


def prepare(case, seed):
    params, inputs = _inputs(case, seed)
    state = dict(case=case, inputs=inputs)
    if case["kind"] == "chunk":
        from smolvla.pipeline import SmolVLAEngine
        engine = SmolVLAEngine(_chunk_config(case), params, case["batch"])
        engine.capture()
        state["engine"] = engine
        return state
    state["params"] = params
    if case["via"] == "graph":
        # the program's static input buffers; new inputs are copied in
        state["static"] = [torch.empty_like(t) for t in inputs]
        state["graph"], state["out"] = _captured(state)
    return state


def _captured(state):
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for dst, src in zip(state["static"], state["inputs"]):
            dst.copy_(src)
        _layer(state["case"], state["params"], state["static"])
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = _layer(state["case"], state["params"], state["static"])
    return graph, out


# -------------------------------------------------------------------- run ---
def run(state):
    if "engine" in state:
        return state["engine"].run(*state["inputs"])
    if "graph" in state:
        for dst, src in zip(state["static"], state["inputs"]):
            dst.copy_(src)
        state["graph"].replay()
        return state["out"]
    return _layer(state["case"], state["params"], state["inputs"])


def _layer(case, p, x):
    kind = case["kind"]
    if kind == "vit":
        from smolvla.config import VitConfig
        from smolvla.vla.vision_block_bf16 import vision_block
        return vision_block(x[0], p, VitConfig(gelu=case["gelu"]))
    if kind == "text":
        from smolvla.vla.text_encoder_bf16 import text_encoder_forward
        # all but the last row (the state token) see each other
        return text_encoder_forward(x[0], p, mask=case["mask"], prefix_len=case["length"] - 1)
    if kind == "self":
        from smolvla.vla.action_expert_bf16 import action_expert_self_forward
        return action_expert_self_forward(x[0], p)
    if kind == "cross":
        from smolvla.vla.action_expert_bf16 import action_expert_cross_forward
        return action_expert_cross_forward(*x, p)
    if kind == "connector":
        from smolvla.vla.connector_bf16 import connector_block
        return connector_block(x[0], p)
    from smolvla.vla.preprocessing_bf16 import preprocessing_block
    return preprocessing_block(x[0], p)


# ------------------------------------------------------------------- work ---
def _pairs(case_mask, L):
    """(query, key) pairs that a head scores."""
    return L * (L + 1) // 2 if case_mask == "causal" else L * L


def _decoder_work(c, B, L, pairs, cross_ctx=None):
    """(flops, weight elements) of one decoder / expert layer."""
    H, q, kv, inter = c["hidden"], c["q"] * HD, c["kv"] * HD, c["inter"]
    w = H * q + q * H + 3 * H * inter
    flops = 2 * B * L * w + 4 * B * pairs * q
    if cross_ctx is None:
        w += 2 * H * kv
        flops += 2 * B * L * 2 * H * kv
    return flops, w


def _vit_work(images, tokens):
    H, inter = VIT["hidden"], VIT["inter"]
    w = 4 * H * H + 2 * H * inter
    return 2 * images * tokens * w + 4 * images * tokens * tokens * H, w


def work(case):
    kind = case["kind"]
    kvd = DEC["kv"] * HD
    if kind == "chunk":
        B, cams = case["batch"], case["cameras"]
        n = B * cams
        L = cams * 64 + case["lang"] + 1
        H = EXP["hidden"]
        pw = VIT["chans"] * VIT["patch"] ** 2 * VIT["hidden"]
        vf, vw = _vit_work(n, 1024)
        cw = VIT["hidden"] * SHUFFLE ** 2 * DEC["hidden"]
        df, dw = _decoder_work(DEC, B, L, L * L)
        sf, sw = _decoder_work(EXP, B, CHUNK, CHUNK * (CHUNK + 1) // 2)
        xf, xw = _decoder_work(EXP, B, CHUNK, CHUNK * L, L)
        iow = 2 * ACTION * H + 2 * H * H      # the time half of W_time_in is per schedule
        flops = (2 * n * 1024 * pw + VIT["layers"] * vf + 2 * n * 64 * cw + DEC["layers"] * df +
                 8 * 2 * B * L * 2 * kvd * kvd +
                 STEPS * (8 * (sf + xf) + 2 * B * CHUNK * iow))
        weights = pw + VIT["layers"] * vw + cw + DEC["layers"] * dw + 8 * 2 * kvd * kvd + \
            8 * (sw + xw) + iow + case["lang"] * B * DEC["hidden"]
        inputs = n * VIT["chans"] * VIT["image"] ** 2 * 2 + B * (STATE + CHUNK * ACTION) * 4
        return dict(bytes=2 * weights + inputs + B * CHUNK * ACTION * 4, flops=flops)
    if kind == "vit":
        f, w = _vit_work(case["images"], case["tokens"])
        return dict(bytes=2 * (w + 2 * case["images"] * case["tokens"] * VIT["hidden"]), flops=f)
    if kind in ("text", "self", "cross"):
        c = DEC if kind == "text" else EXP
        B, L = case["batch"], case["length"]
        io = 2 * B * L * c["hidden"]
        if kind == "text":
            f, w = _decoder_work(c, B, L, _pairs(case["mask"], L))
            io += B * L * 2 * kvd
        elif kind == "self":
            f, w = _decoder_work(c, B, L, _pairs("causal", L))
        else:
            ctx = case["context"]
            f, w = _decoder_work(c, B, L, L * ctx, ctx)
            w += 2 * kvd * kvd
            f += 2 * B * ctx * 2 * kvd * kvd
            io += B * ctx * 2 * kvd
        return dict(bytes=2 * (w + io), flops=f)
    n = case["images"]
    if kind == "connector":
        K, N, M = VIT["hidden"] * SHUFFLE ** 2, DEC["hidden"], n * 64
        return dict(bytes=2 * (M * K + K * N + M * N), flops=2 * M * N * K)
    K, N, M = VIT["chans"] * VIT["patch"] ** 2, VIT["hidden"], n * 1024
    return dict(bytes=2 * (M * K + K * N + 1024 * N + M * N), flops=2 * M * N * K)


# -------------------------------------------------------------- tolerance ---
def tolerance(case):
    """bf16 results.  Measured against float64 (2-norm): 2.3e-3 to 2.9e-3 for
    a layer's outputs and the patch embedding, 1.7e-3 for the connector and a
    whole chunk's actions; about four times that."""
    return {"rel": 7e-3 if case["kind"] in ("chunk", "connector") else 1e-2}


# ------------------------------------------------------------------ exact ---
def _f64(v):
    if torch.is_tensor(v):
        return v.to(F64)
    if isinstance(v, dict):
        return {k: _f64(x) for k, x in v.items()}
    return v


def _rms(x, g):
    return x / torch.sqrt(x.pow(2).mean(-1, keepdim=True) + RMS_EPS) * g


def _ln(x, g, b):
    m = x.mean(-1, keepdim=True)
    v = (x - m).pow(2).mean(-1, keepdim=True)
    return (x - m) / torch.sqrt(v + LN_EPS) * g + b


def _rope(x, heads):
    B, L, _ = x.shape
    half = HD // 2
    k = torch.arange(half, device=x.device, dtype=F64)
    ang = torch.arange(L, device=x.device, dtype=F64)[:, None] / THETA ** (2 * k / HD)
    c, s = ang.cos()[None, :, None], ang.sin()[None, :, None]
    x = x.view(B, L, heads, HD)
    x1, x2 = x[..., :half], x[..., half:]
    return torch.cat([x1 * c - x2 * s, x2 * c + x1 * s], -1)


def _attend(q, k, v, mask):
    """q [L, hq, D], k / v [Lk, hkv, D] of one sample -> [L, hq * D]."""
    L, hq, D = q.shape
    hkv = k.shape[1]
    q, k, v = q.transpose(0, 1), k.transpose(0, 1), v.transpose(0, 1)
    if hkv != hq:
        k, v = (t.repeat_interleave(hq // hkv, 0) for t in (k, v))
    s = torch.matmul(q, k.transpose(1, 2).contiguous()) / math.sqrt(D)
    if mask is not None:
        s.masked_fill_(mask, float("-inf"))
    return torch.matmul(s.softmax(-1), v.contiguous()).transpose(0, 1).reshape(L, hq * D)


def _mask(kind, L, bidir, device):
    i = torch.arange(L, device=device)[:, None]
    j = torch.arange(L, device=device)[None]
    return (j > i) if kind == "causal" else (j > i) & (j >= bidir)


def _mlp(x, p):
    h = _rms(x, p["W_norm_2"])
    g = h @ p["W_gate"]
    return x + ((g * torch.sigmoid(g)) * (h @ p["W_up"])) @ p["W_down"]


def _exact_decoder(x, p, c, mask, bidir=0):
    B, L, _ = x.shape
    h = _rms(x, p["W_norm_1"])
    q, k = _rope(h @ p["Wq"], c["q"]), _rope(h @ p["Wk"], c["kv"])
    v = (h @ p["Wv"]).view(B, L, c["kv"], HD)
    m = _mask(mask, L, bidir, x.device)
    a = torch.stack([_attend(q[b], k[b], v[b], m) for b in range(B)])
    return _mlp(x + a @ p["Wo"], p), k.reshape(B, L, -1), v.reshape(B, L, -1)


def _exact_cross(x, tk, tv, p, c):
    B, Lc, _ = tk.shape
    q = _rope(_rms(x, p["W_norm_1"]) @ p["Wq"], c["q"])
    k = (tk @ p["Wk_cross"]).view(B, Lc, c["kv"], HD)
    v = (tv @ p["Wv_cross"]).view(B, Lc, c["kv"], HD)
    a = torch.stack([_attend(q[b], k[b], v[b], None) for b in range(B)])
    return _mlp(x + a @ p["Wo"], p)


def _gelu(x, kind):
    if kind == "erf":
        return 0.5 * x * (1 + torch.erf(x / math.sqrt(2)))
    return 0.5 * x * (1 + torch.tanh(math.sqrt(2 / math.pi) * (x + 0.044715 * x ** 3)))


def _exact_vit(x, p, gelu):
    """One image at a time ([T, H]): float64 intermediates stay small."""
    def lin(h, w, b):
        y = h @ p[w]
        return y + p[b] if b in p else y

    T = x.shape[0]
    nh = VIT["heads"]
    h = _ln(x, p["W_norm_1"], p["b_norm_1"])
    q, k, v = (lin(h, "W" + n, "b" + n).view(T, nh, HD) for n in "qkv")
    x = x + lin(_attend(q, k, v, None), "Wo", "bo")
    h = _ln(x, p["W_norm_2"], p["b_norm_2"])
    return x + lin(_gelu(lin(h, "W_up", "b_up"), gelu), "W_down", "b_down")


def _exact_shuffle(x):
    """[n, T, E] -> [n, T / 16, 16 E]: row i of the output is the s x s patch
    of tokens at (i // (g/s), i % (g/s)), row by row."""
    n, T, E = x.shape
    g, s = int(round(math.sqrt(T))), SHUFFLE
    return (x.view(n, g // s, s, g // s, s, E).permute(0, 1, 3, 2, 4, 5)
            .reshape(n, T // s ** 2, s * s * E))


def _exact_patch(img, p):
    n, C, S, _ = img.shape
    P = VIT["patch"]
    G = S // P
    cols = img.view(n, C, G, P, G, P).permute(0, 2, 4, 1, 3, 5).reshape(n, G * G, C * P * P)
    return cols @ p["kernel"].reshape(VIT["hidden"], -1).t() + p["bias"] + p["pos_emb"]


def _exact_chunk(case, params, inputs):
    images, ids, state, noise = inputs
    B, cams = case["batch"], case["cameras"]
    S = VIT["image"]
    patch = _f64(params["patch"])
    vis = []
    for im in images.reshape(B * cams, 1, VIT["chans"], S, S):
        vis.append(_exact_patch(im.to(F64), patch)[0])
    for lp in params["vit"]:
        p = _f64(lp)
        vis = [_exact_vit(x, p, "tanh") for x in vis]
    con = torch.stack([_exact_shuffle(x[None])[0] for x in vis]) @ params["connector"]["W"].to(F64)
    con = con.reshape(B, cams * con.shape[1], -1)
    lang = params["embed"][ids].to(F64) * math.sqrt(DEC["hidden"])
    st = state.to(F64)[:, None] @ params["state"]["W"].to(F64)
    x = torch.cat([con, lang, st], 1)
    bidir = x.shape[1] - 1
    kv = []
    for lp in params["prefix"]:
        x, k, v = _exact_decoder(x, _f64(lp), DEC, "prefix_lm", bidir)
        kv.append((k, v))
    io = _f64(params["expert_io"])
    layers = [_f64(lp) for lp in params["expert"]]
    H = EXP["hidden"]
    period = 4e-3 * 1000.0 ** torch.linspace(0, 1, H // 2, dtype=F64, device=x.device)
    xt, t, dt = noise.to(F64), 1.0, -1.0 / STEPS
    for _ in range(STEPS):
        a = xt @ io["W_action_in"] + io["b_action_in"]
        ang = 2 * math.pi * t / period
        te = torch.cat([ang.sin(), ang.cos()]).expand(B, CHUNK, H)
        h = torch.cat([a, te], 2) @ io["W_time_in"] + io["b_time_in"]
        h = (h * torch.sigmoid(h)) @ io["W_time_out"] + io["b_time_out"]
        for i, p in enumerate(layers):
            if i % 2:
                h = _exact_cross(h, *kv[i], p, EXP)
            else:
                h = _exact_decoder(h, p, EXP, "causal")[0]
        xt = xt + dt * (_rms(h, io["W_exp_norm"]) @ io["W_action_out"])
        t += dt
    return xt


def exact(case, seed):
    kind = case["kind"]
    if kind == "chunk" and case["batch"] > 8:
        return None                         # minutes in float64
    params, inputs = _inputs(case, seed)
    if kind == "chunk":
        return _exact_chunk(case, params, inputs)
    p = _f64(params)
    x = inputs[0]
    if kind == "vit":
        return torch.stack([_exact_vit(im.to(F64), p, case["gelu"]) for im in x])
    if kind == "text":
        return _exact_decoder(x.to(F64), p, DEC, case["mask"], case["length"] - 1)
    if kind == "self":
        return _exact_decoder(x.to(F64), p, EXP, "causal")[0]
    if kind == "cross":
        return _exact_cross(x.to(F64), inputs[1].to(F64), inputs[2].to(F64), p, EXP)
    if kind == "connector":
        return torch.stack([_exact_shuffle(im[None].to(F64))[0] @ p["W"] for im in x])
    return torch.stack([_exact_patch(im[None].to(F64), p)[0] for im in x])
