"""The work that programs have this framework do, as cases that can be timed and checked.

A case is a dict of plain values: `kind` names the path, the rest its sizes and options.
listed() gives the standing ones, draw() more of the same ranges.  prepare() makes what a
program holds before the call (registered weights, a model with its KV cache, device
inputs), run() is one pass through the public entry points, exact() the same in 64 bits
from the weight bytes, in plain torch.

Every pass of every state runs on one stream, as a serving loop's calls do; each state has
a context of its own, since the KV cache belongs to the context.
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.abspath("encoding-experiment_amd"))
import larql_hip  # noqa: E402
from larql_hip import F32, Q4_0, Q4_K, Q4_KF, Q6_K, Q8_0  # noqa: E402

FORMATS = {"q4_0": Q4_0, "q4_k": Q4_K, "q4_kf": Q4_KF, "q6_k": Q6_K, "q8_0": Q8_0}
BLOCK = {"q4_0": (32, 18), "q4_k": (256, 148), "q4_kf": (256, 144), "q6_k": (256, 210), "q8_0": (32, 36)}

# Layer geometries: the Llama-3-8B shape of the benchmark's decode and prompt workloads,
# and the [10240 x 2560] geometry of its gate-KNN and walk-FFN workloads as a layer with
# GELU, post-norms, offset norm weights and a sliding window on every layer but the last.
SHAPES = {
    "8b": dict(hidden=4096, inter=14336, nq=32, nkv=8, hd=128, rope=500000.0, vocab=128256, post=False, window=0),
    "4b": dict(hidden=2560, inter=10240, nq=8, nkv=4, hd=256, rope=10000.0, vocab=65536, post=True, window=1024),
}
# Weight formats of a model's projections: all Q4_K; the Q4_K_M mix (V and down in Q6_K);
# Q8_0 attention with Q4_0 FFN (the walk-FFN files).
MIXES = {
    "q4_k": {},
    "q4_k_m": {"wv": "q6_k", "down": "q6_k"},
    "q8_q4_0": {"wq": "q8_0", "wk": "q8_0", "wv": "q8_0", "wo": "q8_0", "gate": "q4_0", "up": "q4_0", "down": "q4_0"},
}


def listed():
    return [
        # one FFN projection of one token: the smallest call, bound by launch and latency
        {"name": "matvec_q4k_ffn", "kind": "matvec", "fmt": "q4_k", "rows": 14336, "cols": 4096, "m": 1},
        # the same projection for a short prompt's six positions
        {"name": "matmul_q4k_6", "kind": "matvec", "fmt": "q4_k", "rows": 14336, "cols": 4096, "m": 6},
        # and for a 512-token prompt at the benchmark's prefill shape
        {"name": "matmul_q4k_512", "kind": "matvec", "fmt": "q4_k", "rows": 10240, "cols": 2560, "m": 512},
        # walk FFN: gate and up scores of a prompt's positions, one layer
        {"name": "pair_q4_0_6", "kind": "pair", "rows": 10240, "cols": 2560, "seq": 6},
        # f32 gate walk over all layers: one query (a token at a time), and a batch
        {"name": "knn_f32_1", "kind": "knn", "fmt": "f32", "layers": 34, "rows": 10240, "cols": 2560, "nq": 1, "k": 10},
        {"name": "knn_f32_256", "kind": "knn", "fmt": "f32", "layers": 34, "rows": 10240, "cols": 2560, "nq": 256, "k": 32},
        # the quantized gate walk, batched
        {"name": "knn_q4_256", "kind": "knn", "fmt": "q4_0", "layers": 34, "rows": 10240, "cols": 2560, "nq": 256, "k": 32},
        # decoding one token: four layers and the vocabulary head, at a chat's and at a long document's position
        {"name": "decode_2k", "kind": "decode", "shape": "8b", "mix": "q4_k", "layers": 4, "pos": 2048},
        {"name": "decode_16k", "kind": "decode", "shape": "8b", "mix": "q4_k", "layers": 4, "pos": 16384},
        # reading a prompt: two layers at 512 positions, a short question in the Q4_K_M mix,
        # and the Q8_0 / Q4_0 layers of walk-FFN files
        {"name": "prompt_512", "kind": "prompt", "shape": "8b", "mix": "q4_k", "layers": 2, "seq": 512},
        {"name": "prompt_24", "kind": "prompt", "shape": "8b", "mix": "q4_k_m", "layers": 2, "seq": 24},
        {"name": "prompt_q4_0_96", "kind": "prompt", "shape": "8b", "mix": "q8_q4_0", "layers": 2, "seq": 96},
    ]


def _log(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["matvec", "matvec", "matmul", "pair", "vecmat", "knn", "knn", "lm_head", "sgemm", "decode",
                       "decode", "prompt", "prompt"])
    if kind == "matvec":  # single activations of every format, small batches of the Q8-input ones
        fmt = rng.choice(["q4_k", "q4_k", "q6_k", "q8_0", "q4_0", "q4_kf"])
        m = _log(rng, 1, 8) if fmt in ("q8_0", "q4_0") else 1
        return {"kind": "matvec", "fmt": fmt, "rows": _log(rng, 1000, 32768), "cols": 256 * rng.randint(4, 56), "m": m}
    if kind == "matmul":  # a prompt's positions through one projection
        return {"kind": "matvec", "fmt": rng.choice(["q4_k", "q4_k", "q6_k"]), "rows": _log(rng, 1000, 16384),
                "cols": 256 * rng.randint(4, 32), "m": _log(rng, 2, 700)}
    if kind == "pair":
        return {"kind": "pair", "rows": _log(rng, 2000, 16384), "cols": 64 * rng.randint(16, 64), "seq": _log(rng, 1, 128)}
    if kind == "vecmat":
        return {"kind": "vecmat", "rows": _log(rng, 2000, 16384), "cols": 32 * rng.randint(32, 128)}
    if kind == "knn":
        return {"kind": "knn", "fmt": rng.choice(["f32", "f32", "q4_0"]), "layers": rng.randint(1, 24),
                "rows": _log(rng, 2000, 12000), "cols": 64 * rng.randint(16, 48), "nq": _log(rng, 1, 256),
                "k": rng.choice([5, 10, 32, 64])}
    if kind == "lm_head":
        return {"kind": "lm_head", "rows": _log(rng, 30000, 130000), "cols": 256 * rng.randint(8, 16),
                "nq": rng.choice([1, 1, 2, 5]), "k": rng.choice([1, 5, 40])}
    if kind == "sgemm":  # f32 products of the trait: one vector to a batch against a matrix
        return {"kind": "sgemm", "m": _log(rng, 1, 512), "kk": rng.randint(500, 2600), "n": _log(rng, 500, 12000),
                "transpose_b": rng.random() < 0.6}
    if kind == "decode":
        return {"kind": "decode", "shape": rng.choice(["8b", "4b"]), "mix": rng.choice(["q4_k", "q4_k_m", "q8_q4_0"]),
                "layers": 4, "pos": _log(rng, 1, 16384)}
    return {"kind": "prompt", "shape": rng.choice(["8b", "4b"]), "mix": rng.choice(["q4_k", "q4_k_m", "q8_q4_0"]),
            "layers": 2, "seq": _log(rng, 2, 512)}


# ── weights in the reference byte layouts ──────────────────────────────────
def _u8(t):
    return t.to(torch.uint8)


def _halves(t):  # f16 values -> their two bytes
    return t.to(torch.float16).contiguous().view(torch.uint8).view(*t.shape, 2)


def _nibbles(q):  # [..., 2n] codes -> n bytes, even element low
    return _u8(q[..., 0::2]) | (_u8(q[..., 1::2]) << 4)


def _fit(x, scale):  # codes of x at a step that may be zero
    return torch.where(scale > 0, x / torch.where(scale > 0, scale, torch.ones_like(scale)), torch.zeros_like(x)).round()


def _quantize(w, fmt):
    """Weights [rows, cols] -> reference bytes (Q8_0: int8 values and f32 scales)."""
    if fmt == "q8_0":
        b = w.view(-1, 32)
        s = b.abs().amax(1, keepdim=True) / 127
        return _fit(b, s).to(torch.int8).view(w.shape), s.view(w.shape[0], -1).contiguous()
    if fmt == "q4_0":
        b = w.view(-1, 32)
        s = (b.abs().amax(1, keepdim=True) / 7).half().float()
        return torch.cat([_halves(s).view(-1, 2), _nibbles(_fit(b, s).clamp(-8, 7) + 8)], 1).view(-1)
    if fmt == "q6_k":
        b = w.view(-1, 16, 16)
        d = (b.abs().amax((1, 2)) / (31 * 32)).half().float()
        sc = _fit(b.abs().amax(2) / 31, d[:, None]).clamp(0, 127)
        q = _fit(b, (d[:, None] * sc)[..., None]).clamp(-32, 31).add(32).view(-1, 256).to(torch.int32)
        hi = (q >> 4).view(-1, 64, 4)
        qh = hi[..., 0] | (hi[..., 1] << 2) | (hi[..., 2] << 4) | (hi[..., 3] << 6)
        return torch.cat([_nibbles(q & 15), _u8(qh), sc.to(torch.int8).view(torch.uint8), _halves(d).view(-1, 2)], 1).view(-1)
    b = w.view(-1, 8, 32)  # q4_k, q4_kf
    lo = b.amin(2).clamp(max=0)
    span = (b.amax(2) - lo) / 15
    top = 15 if fmt == "q4_k" else 63
    d = (span.amax(1) / 63).half().float()
    dm = (-lo.amin(1) / top).half().float()
    sc = _fit(span, d[:, None]).clamp(0, 63)
    mn = _fit(-lo, dm[:, None]).clamp(0, top)
    q = _fit(b + (dm[:, None] * mn)[..., None], (d[:, None] * sc)[..., None]).clamp(0, 15)
    head = torch.cat([_halves(d).view(-1, 2), _halves(dm).view(-1, 2)], 1)
    sc, mn = _u8(sc), _u8(mn)
    if fmt == "q4_k":
        pad = torch.zeros(b.shape[0], 4, dtype=torch.uint8, device=w.device)
        return torch.cat([head, sc, pad, mn[:, :4] | (mn[:, 4:] << 4), _nibbles(q).view(-1, 128)], 1).view(-1)
    packed = torch.cat([(sc[:, :4] & 63) | ((sc[:, 4:] >> 4) << 6), (mn[:, :4] & 63) | ((mn[:, 4:] >> 4) << 6),
                        (sc[:, 4:] & 15) | ((mn[:, 4:] & 15) << 4)], 1)
    q = _u8(q).view(-1, 4, 2, 32)  # a 32-byte chunk: sub-block 2c low, 2c + 1 high
    return torch.cat([head, packed, (q[:, :, 0] | (q[:, :, 1] << 4)).view(-1, 128)], 1).view(-1)


def _values(raw, fmt, rows, cols):
    """The 64-bit values [rows, cols] of reference bytes."""
    if fmt == "q8_0":
        q, s = raw
        return (q.double().view(rows, -1, 32) * s.double()[..., None]).view(rows, cols)
    per, size = BLOCK[fmt]
    b = raw.view(-1, size)
    half = lambda at: b[:, at:at + 2].contiguous().view(torch.float16).double()  # noqa: E731
    both = lambda n: torch.stack([n & 15, n >> 4], -1).flatten(1).double()  # noqa: E731
    if fmt == "q4_0":
        return ((both(b[:, 2:]) - 8) * half(0)).view(rows, cols)
    if fmt == "q6_k":
        qh = b[:, 128:192]
        hi = torch.stack([(qh >> (2 * i)) & 3 for i in range(4)], -1).flatten(1).double()
        q = both(b[:, :128]) + 16 * hi - 32
        sc = b[:, 192:208].contiguous().view(torch.int8).double() * half(208)
        return (q.view(-1, 16, 16) * sc[..., None]).view(rows, cols)
    d, dm = half(0), half(2)
    if fmt == "q4_k":
        sc, mn = b[:, 4:12] & 63, torch.cat([b[:, 16:20] & 15, b[:, 16:20] >> 4], 1)
        q = both(b[:, 20:]).view(-1, 8, 32)
    else:
        p, m, h = b[:, 4:8], b[:, 8:12], b[:, 12:16]
        sc = torch.cat([p & 63, (h & 15) | ((p >> 6) << 4)], 1)
        mn = torch.cat([m & 63, (h >> 4) | ((m >> 6) << 4)], 1)
        n = b[:, 16:].view(-1, 4, 32)
        q = torch.stack([n & 15, n >> 4], 2).view(-1, 8, 32).double()
    return (q * (d * sc.double())[..., None] - (dm * mn.double())[..., None]).view(rows, cols)


def _q8(x):
    """quantize_to_q8 of rows: int8 codes (halves away from zero) and f32 block scales."""
    b = x.view(x.shape[0], -1, 32)
    s = b.abs().amax(2) / torch.full((), 127.0, dtype=b.dtype, device=b.device)
    inv = torch.where(s > 0, 1 / s, torch.zeros_like(s))
    p = b * inv[..., None]
    q = torch.where(p >= 0, torch.floor(p + 0.5), torch.ceil(p - 0.5)).clamp(-128, 127)
    return q.to(torch.int8).view(x.shape), s.contiguous()


def _q8_values(x):
    q, s = _q8(x)
    return (q.double().view(x.shape[0], -1, 32) * s.double()[..., None]).view(x.shape)


# ── inputs ─────────────────────────────────────────────────────────────────
class _Draws:
    """Normal tensors on the GPU from one seed."""

    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda")
        self.gen.manual_seed(seed)

    def normal(self, *shape, std=1.0):
        return torch.randn(*shape, generator=self.gen, device="cuda") * std

    def weight(self, fmt, rows, cols):
        if fmt == "f32":
            return self.normal(rows, cols, std=0.02)
        return _quantize(self.normal(rows, cols, std=0.02), fmt)


def _activations(case, g):
    """A matvec's input: f32 rows, or their Q8 codes and scales."""
    x = g.normal(case["m"], case["cols"])
    return _q8(x) if case["fmt"] in ("q4_0", "q8_0") else (x, None)


NAMES = ("wq", "wk", "wv", "wo", "gate", "up", "down")


def _layer_inputs(case, g):
    """Per layer: projection name -> (format, bytes, rows, cols), the norm vectors, window."""
    s = SHAPES[case["shape"]]
    qd, kvd = s["nq"] * s["hd"], s["nkv"] * s["hd"]
    dims = {"wq": (qd, s["hidden"]), "wk": (kvd, s["hidden"]), "wv": (kvd, s["hidden"]), "wo": (s["hidden"], qd),
            "gate": (s["inter"], s["hidden"]), "up": (s["inter"], s["hidden"]), "down": (s["hidden"], s["inter"])}
    for l in range(case["layers"]):
        ws = {}
        for n in NAMES:
            fmt = MIXES[case["mix"]].get(n, "q4_k")
            ws[n] = (fmt, g.weight(fmt, *dims[n]), *dims[n])
        mean = 0.0 if s["post"] else 1.0
        norms = [g.normal(s["hidden"], std=0.05) + mean for _ in range(4 if s["post"] else 2)]
        yield ws, norms, s["window"] if l + 1 < case["layers"] else 0


def _kv_rows(case, g):
    s = SHAPES[case["shape"]]
    shape = (case["pos"], s["nkv"] * s["hd"])
    return g.normal(*shape).half(), g.normal(*shape).half()


# ── state ──────────────────────────────────────────────────────────────────
_streams = []


def _stream():
    if not _streams:
        _streams.append(torch.cuda.Stream())
    return _streams[0]


class _State:
    """One context with its registered weights or model, and device tensors."""

    def __init__(self, case):
        self.case = case
        self.be = larql_hip.HipBackend(0, strict=True)
        self.model = None
        self.stream = _stream()

    def __del__(self):
        try:
            torch.cuda.synchronize()
            if self.model is not None:
                self.model.close()
            self.be.close()
        except Exception:
            pass

    def register(self, fmt, raw, rows, cols):
        torch.cuda.synchronize()
        if fmt == "f32":
            return self.be.register_weight_device(F32, raw, raw.numel() * 4, rows, cols)
        if fmt == "q8_0":
            return self.be.register_weight_device(Q8_0, raw[0], raw[0].numel(), rows, cols, raw[1])
        return self.be.register_weight_device(FORMATS[fmt], raw, raw.numel(), rows, cols)


def _empty(*shape, dtype=torch.float32):
    return torch.empty(*shape, dtype=dtype, device="cuda")


def _prepare_model(st, g):
    case, s = st.case, SHAPES[st.case["shape"]]
    layers, keep = [], []
    for ws, norms, window in _layer_inputs(case, g):
        keep.append((ws, norms))
        raw = {n: w[1][0] if w[0] == "q8_0" else w[1] for n, w in ws.items()}
        scales = {n: w[1][1] for n, w in ws.items() if w[0] == "q8_0"}
        post = dict(has_post_norms=True, pre_ffn_norm=norms[2], post_ffn_norm=norms[3], norm_offset=1.0,
                    activation=larql_hip.ACT_GELU_TANH) if s["post"] else {}
        layers.append(larql_hip.make_layer(*(raw[n] for n in NAMES), norms[0], norms[1], head_dim=s["hd"],
                                           num_q_heads=s["nq"], num_kv_heads=s["nkv"], rope_base=s["rope"],
                                           formats={n: FORMATS[w[0]] for n, w in ws.items()}, scales=scales,
                                           sliding_window=window, **post))
    torch.cuda.synchronize()
    st.model = st.be.model(layers, s["hidden"], s["inter"], weights_on_device=True)
    del layers, keep
    if case["kind"] == "prompt":
        st.x = g.normal(case["seq"], s["hidden"], std=0.5)
        st.out = _empty(case["seq"], s["hidden"])
        return
    head = g.weight("q6_k", s["vocab"], s["hidden"])
    norm = torch.ones(s["hidden"], device="cuda")
    torch.cuda.synchronize()
    st.model.set_head(head, s["vocab"], norm, fmt=Q6_K, on_device=True)
    for l in range(case["layers"]):
        k, v = _kv_rows(case, g)
        torch.cuda.synchronize()
        st.be.populate_kv_layer_f16_dev(l, k, v, case["pos"], s["nkv"], s["hd"])
    st.x = g.normal(s["hidden"], std=0.5)
    st.out, st.logits = _empty(s["hidden"]), _empty(s["vocab"])


def prepare(case, seed):
    st, g, kind = _State(case), _Draws(seed), case["kind"]
    if kind in ("decode", "prompt"):
        _prepare_model(st, g)
    elif kind == "sgemm":
        m, k, n = case["m"], case["kk"], case["n"]
        st.a, st.b = g.normal(m, k), g.normal(*((n, k) if case["transpose_b"] else (k, n)), std=0.02)
        st.out = _empty(m, n)
    else:
        rows, cols, fmt = case["rows"], case["cols"], case.get("fmt", "q4_0")
        count = case.get("layers", 2 if kind == "pair" else 1)
        st.w = [st.register(fmt, g.weight(fmt, rows, cols), rows, cols) for _ in range(count)]
        if kind == "matvec":
            st.x, st.xs = _activations(case, g)
            st.out = _empty(case["m"], rows)
        elif kind == "pair":
            st.x = g.normal(case["seq"], cols)
            st.out, st.out2 = _empty(case["seq"], rows), _empty(case["seq"], rows)
        elif kind == "vecmat":
            st.x = g.normal(rows)
            st.out = _empty(cols)
        else:  # knn, lm_head
            st.x = g.normal(case["nq"], cols)
            shape = (case["layers"],) if kind == "knn" else ()
            st.idx = _empty(*shape, case["nq"], case["k"], dtype=torch.int32)
            st.val = _empty(*shape, case["nq"], case["k"])
    torch.cuda.synchronize()
    return st


def run(st):
    case, be, s, kind = st.case, st.be, st.stream, st.case["kind"]
    if kind == "matvec":
        be.matvec_dev(st.w[0], st.x, st.out, m=case["m"], x_scales=st.xs, stream=s)
        return st.out
    if kind == "pair":
        be.pair_batch_dev(st.w[0], st.w[1], st.x, case["seq"], st.out, st.out2, stream=s)
        return st.out, st.out2
    if kind == "vecmat":
        be.vecmat_dev(st.w[0], st.x, st.out, stream=s)
        return st.out
    if kind == "knn":
        be.gate_knn_dev(st.w, st.x, case["nq"], case["k"], st.idx, st.val, stream=s)
        return st.idx, st.val
    if kind == "lm_head":
        be.lm_head_knn_dev(st.w[0], st.x, case["nq"], case["k"], st.idx, st.val, stream=s)
        return st.idx, st.val
    if kind == "sgemm":
        be.matmul_dev(st.a, st.b, st.out, case["m"], case["kk"], case["n"], case["transpose_b"], stream=s)
        return st.out
    if kind == "decode":  # the next token at `pos` (the cache rewound to it first)
        be.kv_truncate(case["pos"])
        st.model.decode_dev(st.x, hidden_out=st.out, logits=st.logits, stream=s)
        return st.out, st.logits
    st.model.prefill_dev(st.x, case["seq"], st.out, stream=s)
    return st.out


# ── the work a pass cannot do without ──────────────────────────────────────
def _weight_bytes(fmt, rows, cols):
    if fmt == "f32":
        return 4 * rows * cols
    per, size = BLOCK[fmt]
    return rows * cols // per * size


def _model_work(case):
    s, mix = SHAPES[case["shape"]], MIXES[case["mix"]]
    qd, kvd = s["nq"] * s["hd"], s["nkv"] * s["hd"]
    dims = {"wq": (qd, s["hidden"]), "wk": (kvd, s["hidden"]), "wv": (kvd, s["hidden"]), "wo": (s["hidden"], qd),
            "gate": (s["inter"], s["hidden"]), "up": (s["inter"], s["hidden"]), "down": (s["hidden"], s["inter"])}
    m = case["seq"] if case["kind"] == "prompt" else 1
    by = fl = 0
    for l in range(case["layers"]):
        by += sum(_weight_bytes(mix.get(n, "q4_k"), *d) for n, d in dims.items())
        fl += sum(2 * m * d[0] * d[1] for d in dims.values())
        window = s["window"] if l + 1 < case["layers"] else 0
        if case["kind"] == "prompt":
            w = min(m, window) if window else m
            keys = w * (w + 1) // 2 + (m - w) * w
            by += m * kvd * 2 * 2
        else:
            keys = min(case["pos"] + 1, window) if window else case["pos"] + 1
            by += keys * kvd * 2 * 2
        fl += 4 * keys * qd
    by += 2 * m * s["hidden"] * 4
    if case["kind"] == "decode":
        by += _weight_bytes("q6_k", s["vocab"], s["hidden"]) + 4 * s["vocab"]
        fl += 2 * s["vocab"] * s["hidden"]
    return {"bytes": by, "flops": fl}


def work(case):
    kind = case["kind"]
    if kind in ("decode", "prompt"):
        return _model_work(case)
    if kind == "sgemm":
        m, k, n = case["m"], case["kk"], case["n"]
        return {"bytes": 4 * (m * k + k * n + m * n), "flops": 2 * m * k * n}
    rows, cols, fmt = case["rows"], case["cols"], case.get("fmt", "q4_0")
    wb = _weight_bytes(fmt, rows, cols)
    if kind == "matvec":
        m = case["m"]
        xb = cols * 9 // 8 if fmt in ("q4_0", "q8_0") else 4 * cols
        return {"bytes": wb + m * (xb + 4 * rows), "flops": 2 * m * rows * cols}
    if kind == "pair":
        m = case["seq"]
        return {"bytes": 2 * wb + m * (4 * cols + 8 * rows), "flops": 4 * m * rows * cols}
    if kind == "vecmat":
        return {"bytes": wb + 4 * (rows + cols), "flops": 2 * rows * cols}
    n = case.get("layers", 1)
    return {"bytes": n * wb + case["nq"] * (4 * cols + 8 * n * case["k"]), "flops": 2 * n * case["nq"] * rows * cols}


def tolerance(case):
    kind = case["kind"]
    if kind in ("pair", "knn", "lm_head", "sgemm"):
        return "exact"  # sums in a stated order: block dots in integers, f32 fma chains
    if kind == "matvec":
        if case["fmt"] in ("q4_0", "q8_0"):
            return "exact"
        if case["fmt"] == "q4_k" and case["m"] > 1:
            return {"rel": 1.2e-3, "max": 1e-2}  # operands rounded to fp16 (3e-4 off 64 bits)
        return {"rel": 4e-6, "max": 4e-5}
    if kind == "vecmat":
        return {"rel": 4e-6, "max": 4e-5}
    if case["mix"] == "q8_q4_0":
        # an activation next to a rounding tie takes the neighbouring Q8 code in another order
        # of sums, and what that moves flips more codes in the next layer (7e-3 off 64 bits)
        return {"rel": 3e-2, "max": 3e-1}
    if kind == "decode":
        return {"rel": 2e-5, "max": 2e-4}
    return {"rel": 2e-4, "max": 2e-3}


# ── 64-bit results ─────────────────────────────────────────────────────────
def _rms(x, w, offset):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-6) * (w.double() + offset)


def _rope(x, heads, hd, base, p0):
    n = x.shape[0]
    h = x.view(n, heads, hd)
    i = torch.arange(hd // 2, device=x.device, dtype=torch.float64)
    a = (torch.arange(n, device=x.device, dtype=torch.float64) + p0)[:, None] * base ** (-2 * i / hd)
    c, s = torch.cos(a)[:, None], torch.sin(a)[:, None]
    u, v = h[..., :hd // 2], h[..., hd // 2:]
    return torch.cat([u * c - v * s, u * s + v * c], -1)


def _attend(q, k, v, pos, window, scale):
    """q [n, heads, hd] at positions pos ..; k, v [T, kv, hd]: causal, the last `window` keys."""
    n, heads, hd = q.shape
    at = torch.arange(n, device=q.device)[:, None] + pos
    t = torch.arange(k.shape[0], device=q.device)[None]
    hidden = (t > at) | ((t <= at - window) if window else torch.zeros_like(t > at))
    out = torch.empty_like(q)
    for h in range(heads):
        kv = h // (heads // k.shape[1])
        s = (q[:, h] @ k[:, kv].T * scale).masked_fill(hidden, float("-inf"))
        out[:, h] = torch.softmax(s, 1) @ v[:, kv]
    return out.reshape(n, heads * hd)


def _layer(h, ws, norms, window, s, past, pos):
    def proj(x, n):
        fmt, raw, rows, cols = ws[n]
        x = _q8_values(x) if fmt == "q8_0" or (fmt == "q4_0" and n != "down") else x
        return x @ _values(raw, fmt, rows, cols).T

    off = 1.0 if s["post"] else 0.0
    x = _rms(h, norms[0], off)
    q = _rope(proj(x, "wq"), s["nq"], s["hd"], s["rope"], pos)
    k = _rope(proj(x, "wk"), s["nkv"], s["hd"], s["rope"], pos).half().double()
    v = proj(x, "wv").view(-1, s["nkv"], s["hd"]).half().double()
    if past is not None:
        old = [p.double().view(-1, s["nkv"], s["hd"]) for p in past]
        k, v = torch.cat([old[0], k]), torch.cat([old[1], v])
    o = proj(_attend(q, k, v, pos, window, 1 / math.sqrt(s["hd"])), "wo")
    h = h + (_rms(o, norms[1], off) if s["post"] else o)
    x = _rms(h, norms[2] if s["post"] else norms[1], off)
    g = proj(x, "gate")
    g = torch.nn.functional.gelu(g, approximate="tanh") if s["post"] else torch.nn.functional.silu(g)
    o = proj(g * proj(x, "up"), "down")
    return h + (_rms(o, norms[3], off) if s["post"] else o)


def _exact_model(case, g):
    s = SHAPES[case["shape"]]
    layers = list(_layer_inputs(case, g))
    if case["kind"] == "prompt":
        h = g.normal(case["seq"], s["hidden"], std=0.5).double()
        for ws, norms, window in layers:
            h = _layer(h, ws, norms, window, s, None, 0)
        return h
    head = g.weight("q6_k", s["vocab"], s["hidden"])
    past = [_kv_rows(case, g) for _ in range(case["layers"])]
    h = g.normal(s["hidden"], std=0.5).double()[None]
    for (ws, norms, window), kv in zip(layers, past):
        h = _layer(h, ws, norms, window, s, kv, case["pos"])
    x = _rms(h, torch.ones(s["hidden"], device="cuda"), 0.0)
    logits = torch.cat([x @ _values(r, "q6_k", s["vocab"] // 8, s["hidden"]).T for r in head.chunk(8)], 1)
    return h[0], logits[0]


def exact(case, seed):
    g, kind = _Draws(seed), case["kind"]
    if kind in ("decode", "prompt"):
        return _exact_model(case, g)
    if kind == "sgemm":
        m, k, n = case["m"], case["kk"], case["n"]
        a, b = g.normal(m, k), g.normal(*((n, k) if case["transpose_b"] else (k, n)), std=0.02)
        return a.double() @ (b.double().T if case["transpose_b"] else b.double())
    rows, cols, fmt = case["rows"], case["cols"], case.get("fmt", "q4_0")
    raws = [g.weight(fmt, rows, cols) for _ in range(case.get("layers", 2 if kind == "pair" else 1))]

    def values(raw):
        return raw.double() if fmt == "f32" else _values(raw, fmt, rows, cols)

    if kind == "matvec":
        x, xs = _activations(case, g)
        if xs is not None:
            x = x.double().view(case["m"], -1, 32) * xs.double()[..., None]
        return x.double().view(case["m"], cols) @ values(raws[0]).T
    if kind == "pair":
        x = _q8_values(g.normal(case["seq"], cols))
        return x @ values(raws[0]).T, x @ values(raws[1]).T
    if kind == "vecmat":
        return g.normal(rows).double() @ values(raws[0])
    x = g.normal(case["nq"], cols)
    x = x.double() if fmt == "f32" else _q8_values(x)
    best = []
    for raw in raws:  # the chosen indices have no 64-bit value: near ties rank either way
        sc = x @ values(raw).T
        top = sc if kind == "lm_head" else sc.abs()
        best.append(sc.gather(1, top.topk(case["k"], 1).indices))
    return None, torch.stack(best) if kind == "knn" else best[0]
