"""Performance cases of the framework: the work a user has it do, at the sizes a user meets.

Six kinds of case, each through a public entry point on device-resident data:

* ``linear``   ``ops.linear``: one linear layer, float32 or quantised weight (the drop-in layer);
* ``sdpa``     ``ops.sdpa``: one attention layer of the LM (grouped-query, causal) or the DiT (no mask);
* ``prefill``  ``DeviceQwen2.prefill``: the LM over a prompt; its last logits and the cache rows;
* ``decode``   ``DeviceQwen2.begin`` + ``step_persistent``: greedy speech tokens from a filled cache;
* ``flow``     ``DeviceDiT.solve``: the 10-step classifier-free-guidance solve, noise to mel;
* ``vocoder``  ``DeviceHiFT.decode``: mel and source to waveform, whole or in windows.

Geometries are the framework's own (``cv3amd.synth``): Qwen2-0.5B, the 22-block DiT, HiFTNet at
base 512, with seeded random weights in the converter's storage profiles.  The model's weights are
one fixed checkpoint; the inputs come from the seed.
"""

import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "cosyvoice3-cpu_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from cv3amd import ops, quant, synth  # noqa: E402
from cv3amd.device import to_device  # noqa: E402
from cv3amd.weights import WeightStore  # noqa: E402

STEPS = 10      # Euler steps of a solve
LAYERS, HIDDEN, HEADS, KV_HEADS, HEAD_DIM, INTER = 24, 896, 14, 2, 64, 4864
CAP = 1024      # KV cache rows
PROFILES = ("per_channel", "balanced", "tiny")          # LM storage: int8 per row, int8 block 64, 4-bit body
SHAPES = ((896, 1152), (896, 9728), (4864, 896), (1024, 3072), (1024, 1024), (1024, 2048), (2048, 1024))
WEIGHTS = ("f32", "q8", "q8_rows", "q4")                # of a linear: float32, block 64, per output row, 4-bit


def listed():
    return [
        # one row through a quantised LM projection: the smallest call, all latency
        dict(name="linear 1 row q8", kind="linear", m=1, k=896, n=1152, weight="q8"),
        # a DiT feed-forward layer over both guidance rows of 3.3 s, float32 weights
        dict(name="linear 331 rows f32", kind="linear", m=331, k=1024, n=2048, weight="f32"),
        # the same kind of layer on a converted checkpoint, over 30 s
        dict(name="linear 3000 rows q8", kind="linear", m=3000, k=1024, n=3072, weight="q8"),
        # the LM's attention over a prompt: 14 query heads on 2 key heads, causal
        dict(name="sdpa causal 333", kind="sdpa", heads=14, kv_heads=2, n=333, past=0, causal=True),
        # a short prompt: time to the first token of a sentence
        dict(name="prefill 37 balanced", kind="prefill", t=37, pos0=0, profile="balanced"),
        # a long voice prompt with its text, per-row int8
        dict(name="prefill 500 per_channel", kind="prefill", t=500, pos0=0, profile="per_channel"),
        # speech tokens from a part-filled cache, the LM's token loop
        dict(name="decode 24 from 300", kind="decode", tokens=24, pos=300, profile="per_channel"),
        # a short sentence with float32 weights: 3 s of mel, an odd length
        dict(name="flow 151 f32", kind="flow", t=151, weights="f32"),
        # a whole 10 s segment, float32 weights
        dict(name="flow 500 f32", kind="flow", t=500, weights="f32"),
        # a 30 s segment on the converter's default profile
        dict(name="flow 1500 balanced", kind="flow", t=1500, weights="balanced"),
        # streaming: 1.1 s of mel whole
        dict(name="vocoder 55", kind="vocoder", t=55, chunk=0),
        # a 10 s utterance in 1 s windows
        dict(name="vocoder 500 windows", kind="vocoder", t=500, chunk=50),
    ]


def draw(rng):
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["linear", "linear", "sdpa", "prefill", "decode", "flow", "vocoder"])
    if kind == "linear":
        k, n = rng.choice(SHAPES)
        return dict(kind=kind, m=log_int(1, 3000), k=k, n=n, weight=rng.choice(WEIGHTS))
    if kind == "sdpa":
        if rng.random() < 0.5:
            return dict(kind=kind, heads=16, kv_heads=16, n=log_int(20, 1500), past=0, causal=False)
        n = log_int(8, 800)
        return dict(kind=kind, heads=HEADS, kv_heads=KV_HEADS, n=n, past=rng.choice([0, rng.randint(1, 200)]),
                    causal=True)
    if kind == "prefill":
        t = log_int(5, 800)
        return dict(kind=kind, t=t, pos0=rng.choice([0, rng.randint(1, 200)]), profile=rng.choice(PROFILES))
    if kind == "decode":
        return dict(kind=kind, tokens=rng.randint(4, 40), pos=log_int(20, 900), profile=rng.choice(PROFILES))
    if kind == "flow":
        return dict(kind=kind, t=log_int(40, 1400), weights=rng.choice(["f32", "balanced", "per_channel"]))
    t = log_int(20, 700)
    return dict(kind=kind, t=t, chunk=rng.choice([0, 50, 100]))


# ----------------------------------------------------------------------------------------------
# inputs, weights and handles
# ----------------------------------------------------------------------------------------------

_STORES = {}    # the checkpoint's tensors in host memory, as a program that has read its file holds them


def _store(model, profile):
    if (model, profile) not in _STORES:
        if model == "lm":
            tensors, meta = synth.qwen2_tensors(layers=LAYERS), synth.qwen2_meta(layers=LAYERS)
        elif model == "dit":
            if profile != "f32":
                tensors, meta = _STORES.setdefault("dit raw", synth.dit_tensors()), synth.dit_meta()
            else:
                tensors = _STORES.setdefault("dit raw", synth.dit_tensors())
                meta = synth.dit_meta()
        else:
            tensors, meta = synth.hift_tensors(base=512), synth.hift_meta()
        if profile != "f32":
            tensors = synth.quantize_store(tensors, profile, quant.quantize_q8, quant.quantize_q4)
        _STORES[model, profile] = WeightStore(dict(tensors), meta, quant.QTensor)
    return _STORES[model, profile]


class _Memory:
    """A device array's memory for torch, without a copy."""

    def __init__(self, a):
        self.array = a
        self.__cuda_array_interface__ = {"shape": a.shape, "typestr": a.dtype.str, "data": (a.ptr, False),
                                         "strides": None, "version": 2}


def _tensor(a):
    return torch.as_tensor(_Memory(a), device="cuda")


def _normal(rng, shape, scale=1.0):
    a = rng.standard_normal(shape, dtype=np.float32)
    return a if scale == 1.0 else a * np.float32(scale)


def _linear_inputs(case, seed):
    rng = np.random.default_rng([seed, 1])
    m, k, n = case["m"], case["k"], case["n"]
    x, w, bias = _normal(rng, (m, k)), _normal(rng, (n, k), 0.02), _normal(rng, (n,), 0.02)
    kind = case["weight"]
    if kind == "f32":
        w.flags.writeable = False
        return x, w, bias
    if kind == "q4":
        q, s, _ = quant.quantize_q4(w)
        return x, quant.QTensor("q4", q, s, (n, k), 32), bias
    block = k if kind == "q8_rows" else 64
    q, s, _ = quant.quantize_q8(w, block, np.float32 if kind == "q8_rows" else np.float16)
    return x, quant.QTensor("q8", q, s, (n, k), block), bias


def _sdpa_inputs(case, seed):
    rng = np.random.default_rng([seed, 2])
    h, hk, n, m = case["heads"], case["kv_heads"], case["n"], case["n"] + case["past"]
    return _normal(rng, (h, n, HEAD_DIM)), _normal(rng, (hk, m, HEAD_DIM)), _normal(rng, (hk, m, HEAD_DIM))


def _lm_inputs(case, seed):
    """Embeddings of a prompt and the cache rows before it."""
    rng = np.random.default_rng([seed, 3])
    past = case["pos0"] if case["kind"] == "prefill" else case["pos"]
    k, v = (_normal(rng, (LAYERS, KV_HEADS, past, HEAD_DIM)) for _ in range(2))
    if case["kind"] == "prefill":
        return k, v, _normal(rng, (case["t"], HIDDEN), 0.5)
    return k, v, int(rng.integers(0, synth.SPEECH_TOKEN_SIZE))


def _flow_inputs(case, seed):
    rng = np.random.default_rng([seed, 4])
    t = case["t"]
    return (_normal(rng, (1, 80, t)), _normal(rng, (1, 80)), _normal(rng, (1, 80, t)), _normal(rng, (1, 80, t)))


def _vocoder_inputs(case, seed):
    rng = np.random.default_rng([seed, 5])
    t = case["t"]
    mel = rng.normal(-5.0, 2.0, (80, t)).astype(np.float32)
    f0 = 120.0 + 60.0 * np.sin(np.arange(480 * t) * (2 * math.pi / 24000 * 1.7))
    source = 0.1 * np.sin(2 * math.pi * np.cumsum(f0) / 24000) + 0.003 * rng.standard_normal(480 * t)
    return mel, source.astype(np.float32)


def prepare(case, seed):
    kind, s = case["kind"], {"case": case}
    if kind == "linear":
        x, s["w"], bias = _linear_inputs(case, seed)
        bias.flags.writeable = False
        s["x"], s["bias"] = to_device(x), bias
        ops.linear(s["x"], s["w"], bias)    # the layer's weights go to the device with the first call
    elif kind == "sdpa":
        s["q"], s["k"], s["v"] = (to_device(a) for a in _sdpa_inputs(case, seed))
    elif kind in ("prefill", "decode"):
        from cv3amd.qwen2 import DeviceQwen2
        k, v, first = _lm_inputs(case, seed)
        lm = s["lm"] = DeviceQwen2(_store("lm", case["profile"]), cap=CAP)
        if k.shape[2]:
            lm.fill_cache(k, v)
        s["first"] = to_device(first) if kind == "prefill" else first
        # the program's view of what the LM writes
        s["out"] = [_tensor(lm.logits), _tensor(lm.k_cache), _tensor(lm.v_cache), _tensor(lm.ints)]
    elif kind == "flow":
        from cv3amd.dit import DeviceDiT
        mu, spks, cond, s["x0"] = _flow_inputs(case, seed)
        s["dit"] = DeviceDiT(_store("dit", case["weights"]), steps=STEPS)
        s["dit"].prepare(mu, spks, cond)
    else:
        from cv3amd.hift import DeviceHiFT
        mel, source = _vocoder_inputs(case, seed)
        s["hift"] = DeviceHiFT(_store("hift", "f32"))
        s["mel"], s["source"] = to_device(mel), to_device(source)
    return s


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "linear":
        return _tensor(ops.linear(s["x"], s["w"], s["bias"]))
    if kind == "sdpa":
        mask = ("causal", case["past"]) if case["causal"] else None
        return _tensor(ops.sdpa(s["q"], s["k"], s["v"], mask))
    if kind == "prefill":
        s["lm"].prefill(s["first"], case["pos0"])
        return s["out"][:3]
    if kind == "decode":
        lm = s["lm"]
        lm.begin(s["first"], case["pos"])
        for _ in range(case["tokens"]):
            lm.step_persistent()
        return s["out"]
    if kind == "flow":
        return _tensor(s["dit"].solve(s["x0"], graph=True))
    return _tensor(s["hift"].decode(s["mel"], s["source"], chunk=case["chunk"] or None))


# ----------------------------------------------------------------------------------------------
# what a pass cannot do without
# ----------------------------------------------------------------------------------------------

_BITS = {"f32": 4.0, "q8": 1.0 + 2.0 / 64, "q8_rows": 1.0, "per_channel": 1.0, "balanced": 1.0 + 2.0 / 64,
         "q4": 0.5 + 2.0 / 32, "tiny": 0.5 + 2.0 / 32}                    # bytes per weight


def _hift_convs(t):
    """(weights, multiply-adds) of the vocoder's convs over t mel frames."""
    m = synth.HIFT_META
    rates, base = m["upsample_rates"], 512
    down = [int(np.prod([1] + rates[::-1][:i])) for i in range(1, 4)][::-1]
    total, weights, now = 0, 0, t

    def add(cin, cout, k, rows):
        nonlocal total, weights
        total += cin * cout * k * rows
        weights += cin * cout * k

    add(80, base, 5, t)
    for i, r in enumerate(rates):
        now *= r
        cin, c = base >> i, base >> (i + 1)
        add(cin, c, m["upsample_kernel_sizes"][i], now)
        add(18, c, 2 * down[i] if down[i] > 1 else 1, now)
        for k in [m["source_resblock_kernel_sizes"][i]] + m["resblock_kernel_sizes"]:
            for _ in range(6):
                add(c, c, k, now)
    add(base // 8, 18, 7, now)
    return weights, total


def work(case):
    kind = case["kind"]
    if kind == "linear":
        m, k, n = case["m"], case["k"], case["n"]
        return {"bytes": 4.0 * m * (k + n) + _BITS[case["weight"]] * n * k, "flops": 2.0 * m * n * k}
    if kind == "sdpa":
        h, hk, n, m = case["heads"], case["kv_heads"], case["n"], case["n"] + case["past"]
        pairs = n * case["past"] + n * (n + 1) / 2 if case["causal"] else n * m
        return {"bytes": 4.0 * HEAD_DIM * (2 * h * n + 2 * hk * m), "flops": 4.0 * h * HEAD_DIM * pairs}
    if kind in ("prefill", "decode"):
        body = LAYERS * HIDDEN * ((HEADS + 2 * KV_HEADS) * HEAD_DIM + HIDDEN + 3 * INTER)
        head = HIDDEN * synth.LM_HEAD_ROWS
        t, past = (case["t"], case["pos0"]) if kind == "prefill" else (case["tokens"], case["pos"])
        per_w, kv = _BITS[case["profile"]], 2 * 4.0 * LAYERS * KV_HEADS * HEAD_DIM
        pairs = t * past + t * (t + 1) / 2
        attention = 4.0 * LAYERS * HEADS * HEAD_DIM * pairs
        if kind == "prefill":
            return {"bytes": per_w * body + head + kv * (past + 2 * t) + 4.0 * HIDDEN * t,
                    "flops": 2.0 * body * t + 2.0 * head + attention}
        return {"bytes": t * (per_w * body + head) + kv * (pairs + t), "flops": 2.0 * t * (body + head) + attention}
    if kind == "flow":
        t, d, depth = case["t"], 1024, 22
        weights = depth * 8 * d * d
        edges = 4 * 80 * d + 80 * d + 2 * d * 64 * 31
        per_step = 2.0 * 2 * t * (weights + edges) + depth * 4.0 * 2 * t * t * d
        mods = (6 * depth + 2) * d * d
        per_w = _BITS[case["weights"]]
        # one step's weights are read each step (they do not stay on the chip)
        return {"bytes": STEPS * (per_w * weights + 4.0 * edges) + per_w * mods + 4.0 * 5 * 80 * t,
                "flops": STEPS * (per_step + 2.0 * mods)}
    weights, macs = _hift_convs(case["t"])
    return {"bytes": 4.0 * weights + 4.0 * case["t"] * (80 + 2 * 480), "flops": 2.0 * macs}


def tolerance(case):
    """About four times the measured distance of the float32 results from the 64-bit ones (linear and
    sdpa 2e-7 to 1e-6, prefill 3e-6, decode 1.3e-6, flow 1.3e-7, vocoder 1e-6), with room for another
    implementation's own error of that size."""
    return {"linear": {"rel": 4e-6, "max": 1e-4},
            "sdpa": {"rel": 4e-6, "max": 1e-4},
            "prefill": {"rel": 1e-5, "max": 4e-4},
            "decode": {"rel": 1e-5, "max": 4e-4, "differ": 0.0},
            "flow": {"rel": 1e-6, "max": 5e-5},
            "vocoder": {"rel": 8e-6, "max": 8e-4}}[case["kind"]]


# ----------------------------------------------------------------------------------------------
# the same results in 64 bits, from the definitions
# ----------------------------------------------------------------------------------------------

def _d(a):
    return torch.as_tensor(np.ascontiguousarray(a)).cuda().double()


def _weight(w):
    """A stored weight's values: codes times scales for a quantised one."""
    if isinstance(w, np.ndarray):
        return _d(w)
    q, s = np.asarray(w.q), _d(np.asarray(w.scales))
    if w.kind == "q4":      # byte j of a 32-code block holds code j low, code j + 16 high, each + 8
        b = torch.as_tensor(q.astype(np.uint8)).cuda().reshape(q.shape[0], -1, 16)
        q = torch.cat([b & 15, b >> 4], dim=2).double() - 8
    else:
        q = _d(q).reshape(q.shape[0], -1, int(w.block))
    return (q * s[:, :, None]).reshape(q.shape[0], -1)[:, :w.shape[1]].contiguous()


def _attend(q, k, v, past=None):
    """(H, N, D) x (Hk, M, D): softmax(q k^T / sqrt(D)) v, causal after `past` keys unless None."""
    h, n, d = q.shape
    m, rep = k.shape[1], q.shape[0] // k.shape[0]
    out = torch.empty_like(q)
    for i in range(h):
        s = q[i] @ k[i // rep].t().contiguous() / math.sqrt(d)
        if past is not None:
            s.masked_fill_(torch.arange(m, device=s.device)[None] > torch.arange(n, device=s.device)[:, None] + past,
                           -math.inf)
        out[i] = torch.softmax(s, dim=-1) @ v[i // rep]
    return out


def _exact_lm(case, seed):
    ks, vs, first = _lm_inputs(case, seed)
    store = _store("lm", case["profile"])
    past = ks.shape[2]
    kc, vc = (torch.zeros((LAYERS, KV_HEADS, CAP, HEAD_DIM), dtype=torch.float64, device="cuda") for _ in range(2))
    kc[:, :, :past], vc[:, :, :past] = _d(ks), _d(vs)
    half = HEAD_DIM // 2
    inv = 1.0 / (1e6 ** (np.arange(0, HEAD_DIM, 2, dtype=np.float64) / HEAD_DIM))
    ang = np.arange(CAP, dtype=np.float64)[:, None] * inv[None]
    cos, sin = (_d(np.concatenate([f(ang)] * 2, axis=1)) for f in (np.cos, np.sin))
    w = {}

    def get(name):
        if name not in w:
            w[name] = _weight(store.get("llm." + name))
        return w[name]

    def rms(x, name):
        return x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-6) * get(name)

    def forward(h, pos):
        t = h.shape[0]
        c, s = cos[pos:pos + t], sin[pos:pos + t]
        for i in range(LAYERS):
            p = "model.layers.%d." % i
            n = rms(h, p + "input_layernorm")
            q, k, v = ((n @ get(p + "self_attn.%s_proj.weight" % x).t() + get(p + "self_attn.%s_proj.bias" % x))
                       .reshape(t, -1, HEAD_DIM).transpose(0, 1) for x in "qkv")
            q, k = (x * c + torch.cat([-x[..., half:], x[..., :half]], dim=-1) * s for x in (q, k))
            kc[i, :, pos:pos + t], vc[i, :, pos:pos + t] = k, v
            a = _attend(q.contiguous(), kc[i, :, :pos + t], vc[i, :, :pos + t], pos)
            h = h + a.transpose(0, 1).reshape(t, -1) @ get(p + "self_attn.o_proj.weight").t()
            n = rms(h, p + "post_attention_layernorm")
            g = n @ get(p + "mlp.gate_proj.weight").t()
            h = h + (g * torch.sigmoid(g) * (n @ get(p + "mlp.up_proj.weight").t())) @ get(p + "mlp.down_proj.weight").t()
        return rms(h[-1], "model.norm") @ get("llm_decoder.weight").t() + get("llm_decoder.bias")

    if case["kind"] == "prefill":
        return [forward(_d(first), past), kc, vc]
    token, emb = first, _weight(store.get("llm.speech_embedding"))
    for i in range(case["tokens"]):
        logits = forward(emb[token][None], past + i)
        token = int(logits.argmax())
    return [logits, kc, vc, None]


def _exact_flow(case, seed):
    mu, spks, cond, x0 = _flow_inputs(case, seed)
    store, t, d, heads = _store("dit", case["weights"]), case["t"], 1024, 16
    w = {}

    def get(name):
        if name not in w:
            w[name] = _weight(store.get("flow.decoder.estimator." + name))
        return w[name]

    def lin(x, name):
        return x @ get(name + ".weight").t() + get(name + ".bias")

    def norm(x):
        c = x - x.mean(-1, keepdim=True)
        return c / torch.sqrt((c * c).mean(-1, keepdim=True) + 1e-6)

    def conv(x, name):      # (T, 1024): 16 groups, 31 taps back, then Mish
        wt = _d(store.get("flow.decoder.estimator." + name + ".weight"))
        xp = torch.cat([x.new_zeros(30, d), x]).reshape(t + 30, 16, 64).transpose(0, 1)     # (16, T + 30, 64)
        y = x.new_zeros(16, t, 64)
        for k in range(31):
            y += torch.bmm(xp[:, k:k + t].contiguous(), wt[:, :, k].reshape(16, 64, 64).transpose(1, 2).contiguous())
        y = y.transpose(0, 1).reshape(t, d) + get(name + ".bias")
        return y * torch.tanh(torch.nn.functional.softplus(y))

    inv = 1.0 / (10000.0 ** (np.arange(0, 64, 2, dtype=np.float64) / 64))
    ang = _d(np.repeat(np.arange(t, dtype=np.float64)[:, None] * inv[None], 2, axis=-1).astype(np.float32))
    cos, sin = torch.cos(ang), torch.sin(ang)

    def rope(x):            # the first 64 channels, in pairs
        a = x[:, :64]
        turned = torch.stack([-a[:, 1::2], a[:, 0::2]], dim=-1).reshape(t, 64)
        return torch.cat([a * cos + turned * sin, x[:, 64:]], dim=1)

    def split(x):
        return x.reshape(t, heads, 64).transpose(0, 1).contiguous()

    span = (1.0 - np.cos(np.linspace(0.0, 1.0, STEPS + 1, dtype=np.float64) * 0.5 * np.pi)).astype(np.float32)
    freq = np.exp(np.arange(128, dtype=np.float32) * -(math.log(10000.0) / 127))
    x = _d(x0[0])
    now, dt = span[0], span[1] - span[0]
    for step in range(1, STEPS + 1):
        arg = _d(1000.0 * np.asarray(now).reshape(-1, 1).astype(np.float32) * freq[None])
        temb = lin(torch.cat([torch.sin(arg), torch.cos(arg)], dim=-1), "time_embed.time_mlp.0")
        temb = lin(temb * torch.sigmoid(temb), "time_embed.time_mlp.2")
        temb = temb * torch.sigmoid(temb)
        got = []
        for row in range(2):
            on = 1.0 - row
            h = lin(torch.cat([x.t(), on * _d(cond[0].T), on * _d(mu[0].T), on * _d(spks).expand(t, 80)], dim=1),
                    "input_embed.proj")
            h = h + conv(conv(h, "input_embed.conv_pos_embed.conv1.0"), "input_embed.conv_pos_embed.conv2.0")
            for i in range(22):
                b = "transformer_blocks.%d." % i
                sh_a, sc_a, g_a, sh_m, sc_m, g_m = lin(temb, b + "attn_norm.linear").chunk(6, dim=1)
                n = norm(h) * (1.0 + sc_a) + sh_a
                q, k, v = (lin(n, b + "attn.to_" + c) for c in "qkv")
                a = _attend(split(rope(q)), split(rope(k)), split(v)).transpose(0, 1).reshape(t, d)
                h = h + g_a * lin(a, b + "attn.to_out.0")
                n = norm(h) * (1.0 + sc_m) + sh_m
                f = torch.nn.functional.gelu(lin(n, b + "ff.ff.0.0"), approximate="tanh")
                h = h + g_m * lin(f, b + "ff.ff.2")
            scale, shift = lin(temb, "norm_out.linear").chunk(2, dim=1)
            got.append(lin(norm(h) * (1.0 + scale) + shift, "proj_out").t())
        x = x + float(dt) * (1.7 * got[0] - 0.7 * got[1])
        now = now + dt
        if step < STEPS:
            dt = span[step + 1] - now
    return x


def _exact_vocoder(case, seed):
    mel, source = _vocoder_inputs(case, seed)
    store, meta = _store("hift", "f32"), synth.HIFT_META
    get = lambda n: _d(store.get("hift." + n))  # noqa: E731

    def conv(x, name, stride=1, dilation=1, left=0, right=0):
        w = get(name + ".weight")
        k = w.shape[2]
        x = torch.nn.functional.pad(x, (left, right))
        n = (x.shape[1] - dilation * (k - 1) - 1) // stride + 1
        y = x.new_zeros(w.shape[0], n)
        for j in range(k):
            y += w[:, :, j].contiguous() @ x[:, j * dilation:j * dilation + (n - 1) * stride + 1:stride].contiguous()
        return y + get(name + ".bias")[:, None]

    def snake(x, name):
        a = get(name)[:, None]
        return x + torch.sin(a * x) ** 2 / (a + 1e-9)

    def leaky(x, slope):
        return torch.where(x >= 0, x, slope * x)

    def resblock(x, base, k, dilations):
        for j, dil in enumerate(dilations):
            y = conv(snake(x, "%sactivations1.%d.alpha" % (base, j)), "%sconvs1.%d" % (base, j), dilation=dil,
                     left=(k - 1) * dil)
            x = x + conv(snake(y, "%sactivations2.%d.alpha" % (base, j)), "%sconvs2.%d" % (base, j), left=k - 1)
        return x

    n_fft, hop, rates = meta["istft_n_fft"], meta["istft_hop_len"], meta["upsample_rates"]
    win = _d((0.5 - 0.5 * np.cos(2.0 * np.pi * np.arange(n_fft) / n_fft)).astype(np.float32))
    src = _d(np.pad(source, (n_fft // 2, n_fft // 2), mode="reflect")).unfold(0, n_fft, hop) * win
    spec = torch.as_tensor(np.fft.rfft(src.cpu().numpy(), axis=1).T.copy()).cuda()
    spec = torch.cat([spec.real, spec.imag])
    x = conv(_d(mel), "conv_pre", right=4)
    downs = [15, 3, 1]
    for i, r in enumerate(rates):
        k = store.get("hift.ups.%d.weight" % i).shape[2]
        x = conv(leaky(x, meta["lrelu_slope"]).repeat_interleave(r, dim=1), "ups.%d" % i, left=k - 1)
        if i == len(rates) - 1:
            x = torch.cat([x[:, 1:2], x], dim=1)
        u = downs[i]
        s = conv(spec, "source_downs.%d" % i, stride=u, left=u - 1)
        x = x + resblock(s, "source_resblocks.%d." % i, meta["source_resblock_kernel_sizes"][i],
                         meta["source_resblock_dilation_sizes"][i])
        x = sum(resblock(x, "resblocks.%d." % (3 * i + j), meta["resblock_kernel_sizes"][j],
                         meta["resblock_dilation_sizes"][j]) for j in range(3)) / 3.0
    x = conv(leaky(x, 0.01), "conv_post", left=6)
    half = n_fft // 2 + 1
    mag, ph = torch.clamp(torch.exp(torch.clamp(x[:half], max=80.0)), max=1e2).cpu().numpy(), torch.sin(x[half:]).cpu().numpy()
    frames = np.fft.irfft(mag * np.cos(ph) + 1j * mag * np.sin(ph), n=n_fft, axis=0) * win.cpu().numpy()[:, None]
    nfr = frames.shape[1]
    y, env = (np.zeros((nfr - 1) * hop + n_fft) for _ in range(2))
    for j in range(n_fft):
        y[j:j + (nfr - 1) * hop + 1:hop] += frames[j]
        env[j:j + (nfr - 1) * hop + 1:hop] += float(win[j]) ** 2
    y[env > 1e-11] /= env[env > 1e-11]
    return torch.as_tensor(np.clip(y[n_fft // 2:-(n_fft // 2)], -meta["audio_limit"], meta["audio_limit"]))


def exact(case, seed):
    kind = case["kind"]
    if kind == "linear":
        x, w, bias = _linear_inputs(case, seed)
        return _d(x) @ _weight(w).t() + _d(bias)
    if kind == "sdpa":
        q, k, v = (_d(a) for a in _sdpa_inputs(case, seed))
        return _attend(q, k, v, case["past"] if case["causal"] else None)
    if kind in ("prefill", "decode"):
        return _exact_lm(case, seed)
    return _exact_flow(case, seed) if kind == "flow" else _exact_vocoder(case, seed)
