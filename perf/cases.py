"""The calls that programs make of this framework, for timing them: what each needs in hand, one pass, its smallest work.

Shapes are those of the benchmark and the tests: the Bonsai-8B layer (hidden 4096, 32 query / 8 KV heads of 128, FFN
12288, vocabulary 151,936, 36 layers) over Q1_0 weights, and the north-mini-code block (hidden 2048, 32 query / 4 KV
heads of 128, 128 experts of 768, top-8, window 4096 on three layers of four) over Q4_K / Q6_K weights. Activations and
caches are fixed point with 16 fraction bits; Q1_0 scales are the int32 range that 8B checkpoints have (an fp16 scale
near 2^-6 is about 1000) or, for the linear alone, the codec's whole fp16 range (64-bit scales).

Weights are laid out once per process from fixed seeds and kept, as a serving program keeps its model; everything that
a call is given (activations, prompts, caches, routes, gates) comes from the case's seed. Every output is a whole
number and has to be the same to the last bit.
"""
from __future__ import annotations

import ctypes
from types import SimpleNamespace

import numpy as np
import torch

from integer_inference_engine_amd import _lib, gpu_native, qk_gpu
from integer_inference_engine_amd.resident import ResidentNet
from integer_inference_engine_amd.rope_tables import bonsai8b_tables, plain_tables

FRAC = 16
D, H, HKV, HD, DFF, VOCAB, LAYERS = 4096, 32, 8, 128, 12288, 151936, 36
PROJ = {"wq": (H * HD, D), "wk": (HKV * HD, D), "wv": (HKV * HD, D), "wo": (D, H * HD), "w1": (DFF, D),
        "wu": (DFF, D), "w2": (D, DFF)}
LAYER_WEIGHTS = sum(o * i for o, i in PROJ.values())
# north-mini-code
ND, NH, NKV, NHD, EXPERTS, TOP, NFF, WINDOW, FW = 2048, 32, 4, 128, 128, 8, 768, 4096, 24
EXPERT_BYTES = 2 * NFF * (ND // 256) * 144 + ND * (NFF // 256) * 210
ROPE_ROWS = 16384 + 512
REPLY = 128                      # tokens generated on one imported north-mini-code prompt before the next request
INV_SQRT = int(round((1 << FRAC) / float(np.sqrt(HD))))

_kept = {}                       # weights, tables and models laid out once


def _keep(key, make):
    if key not in _kept:
        _kept[key] = make()
    return _kept[key]


# ---- the cases ----------------------------------------------------------------------------------------------------
def listed():
    return [
        # one token through one resident projection: the smallest call, bound by launches and latency
        {"name": "linear_1", "kind": "linear", "tokens": 1, "out": 4096, "inp": 4096, "scale": "i32"},
        # a medium, odd number of rows (a short prompt, a wide batch) against a weight with codec-range 64-bit scales
        {"name": "linear_93_i64", "kind": "linear", "tokens": 93, "out": 4096, "inp": 12288, "scale": "i64"},
        # the reference's own entry points, host arrays in and out over an int64 cache: a prompt in one call with its
        # K/V handed back, then one step of a small batch seeded with such K/V
        {"name": "monolith_256", "kind": "monolith", "tokens": 256, "layers": 12},
        {"name": "ctx_step_4", "kind": "ctx_step", "batch": 4, "layers": 6, "lo": 300, "hi": 1500},
        # prefill into the resident paged cache: a whole long prompt, and an odd chunk behind a long prefix
        {"name": "prefill_2048", "kind": "prefill", "tokens": 2048, "start": 0, "layers": 2},
        {"name": "prefill_333_at_5000", "kind": "prefill", "tokens": 333, "start": 5000, "layers": 2},
        # generation on the device: one interactive sequence through the full model, and a ragged serving batch with
        # the sampler (each pass: one forward that sets the positions, then the decode loop)
        {"name": "generate_1", "kind": "generate", "batch": 1, "layers": 36, "lo": 4096, "hi": 4096, "steps": 8,
         "mode": "greedy"},
        {"name": "generate_32", "kind": "generate", "batch": 32, "layers": 4, "lo": 512, "hi": 16000, "steps": 4,
         "mode": "top_p"},
        # the MoE block for one token and for a batch
        {"name": "moe_1", "kind": "moe", "tokens": 1},
        {"name": "moe_64", "kind": "moe", "tokens": 64},
        # one token through a period of north-mini-code layers (three windowed with RoPE, one full without) on the
        # retained bank: norm, router, attention, experts
        {"name": "nmc_token", "kind": "nmc_token", "context": 4600, "layers": 4},
        # receipt verification of a turn by the full model: teacher-forced logits, re-drawn tokens, row digests
        {"name": "verify_512", "kind": "verify", "tokens": 512, "out": 256},
    ]


def _log(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["linear", "linear", "monolith", "ctx_step", "prefill", "prefill", "generate", "generate", "moe",
                       "moe", "nmc_token", "verify"])
    if kind == "linear":
        out, inp = rng.choice([(4096, 4096), (1024, 4096), (12288, 4096), (4096, 12288), (5000, 2688), (333, 1408)])
        return {"kind": kind, "tokens": _log(rng, 1, 512), "out": out, "inp": inp, "scale": rng.choice(["i32", "i64"])}
    if kind == "monolith":
        return {"kind": kind, "tokens": _log(rng, 8, 400), "layers": rng.choice([2, 6, 12])}
    if kind == "ctx_step":
        lo = _log(rng, 40, 800)
        return {"kind": kind, "batch": rng.randint(1, 6), "layers": 4, "lo": lo, "hi": rng.randint(lo, 1600)}
    if kind == "prefill":
        start = rng.choice([0, 0, _log(rng, 64, 8000)])
        return {"kind": kind, "tokens": _log(rng, 16, 2048 if start == 0 else 1024), "start": start, "layers": 2}
    if kind == "generate":
        batch = _log(rng, 1, 32)
        lo = _log(rng, 64, 8000)
        return {"kind": kind, "batch": batch, "layers": 4, "lo": lo, "hi": rng.randint(lo, 15000),
                "steps": rng.randint(3, 6), "mode": rng.choice(["greedy", "top_p"])}
    if kind == "moe":
        return {"kind": kind, "tokens": _log(rng, 1, 512)}
    if kind == "nmc_token":
        return {"kind": kind, "context": _log(rng, 32, 8000), "layers": 4}
    tokens = _log(rng, 80, 500)
    return {"kind": kind, "tokens": tokens, "out": rng.randint(16, tokens - 16)}


# ---- weights --------------------------------------------------------------------------------------------------------
def _q1_host(out, inp, seed, scale="i32"):
    r = np.random.default_rng(seed)
    bits = r.integers(0, 256, size=(out, inp // 128, 16), dtype=np.uint8)
    if scale == "i32":
        return bits, r.integers(1, 4097, size=(out, inp // 128), dtype=np.int64)
    v = r.integers(0, 0x7C00, size=(out, inp // 128), dtype=np.uint16).view(np.float16).astype(np.float64)
    v = np.where(r.integers(0, 2, size=v.shape) == 1, -v, v)
    return bits, np.rint(v * 65536.0).astype(np.int64)


def _register(bits, scale):
    h = gpu_native.q1_register_weight(bits, scale)
    assert h is not None, _lib.last_error()
    return h


def _upload(a):
    h = gpu_native.buf_upload_i64(a)
    assert h is not None, _lib.last_error()
    return h


def _tables():
    return _keep("tables", lambda: bonsai8b_tables(ROPE_ROWS))


def _model(layers):
    """Handle bundles (w, g) of the 8B-shape model's first `layers` layers with its head, and the embedding."""
    def one_layer():
        proj = {k: _q1_host(o, i, 100 + n) for n, (k, (o, i)) in enumerate(PROJ.items())}
        r = np.random.default_rng(7)
        gains = {k: r.integers(1 << 15, (1 << 17) + 1, size=n, dtype=np.int64)
                 for k, n in (("n1g", D), ("n2g", D), ("qng", HD), ("kng", HD))}
        return proj, gains

    proj, gains = _keep("host_layer", one_layer)
    have = _keep("layers", list)
    while len(have) < layers:    # separately resident layers, as the full model's are
        have.append(({k: _register(*v) for k, v in proj.items()}, {k: _upload(v) for k, v in gains.items()}))

    def head():
        bits, scale = _q1_host(VOCAB, D, 200)
        final = np.random.default_rng(9).integers(1 << 15, (1 << 17) + 1, size=D, dtype=np.int64)
        cos, sin = _tables()
        return {"out_head": _register(bits, scale), "finalg": _upload(final), "cos_h": _upload(cos),
                "sin_h": _upload(sin), "final": final, "bits": bits, "scale": scale,
                "ebits": torch.from_numpy(bits).cuda(), "escale": torch.from_numpy(scale).cuda()}

    t = _keep("head", head)
    w = {k: np.array([x[0][k] for x in have[:layers]], dtype=np.int64) for k in PROJ}
    g = {k: np.array([x[1][k] for x in have[:layers]], dtype=np.int64) for k in ("n1g", "n2g", "qng", "kng")}
    w["out_head"], w["out_head_vocab"] = t["out_head"], VOCAB
    g["finalg"], g["cos_h"], g["sin_h"] = t["finalg"], t["cos_h"], t["sin_h"]
    return w, g, t


def _verifier():
    def make():
        from integer_inference_engine_amd.verify import DeviceVerifier
        proj, gains = _model(1) and _kept["host_layer"]
        head = _kept["head"]
        layer = {"n1_gain_fp": gains["n1g"], "n2_gain_fp": gains["n2g"], "q_norm_gain_fp": gains["qng"],
                 "k_norm_gain_fp": gains["kng"]}
        for k, (bits, scale) in proj.items():
            layer[f"{k}_bits"], layer[f"{k}_scale_fp"] = bits, scale
        cos, sin = _tables()
        config = {"architecture": "qwen3", "dModel": D, "nLayers": LAYERS, "n_heads": H, "n_heads_kv": HKV,
                  "head_dim": HD, "dFfn": DFF, "vocab": VOCAB, "context_len": 2048, "frac": FRAC}
        return DeviceVerifier({"config": config, "embed_bits": head["bits"], "embed_scale_fp": head["scale"],
                               "output_bits": head["bits"], "output_scale_fp": head["scale"],
                               "final_norm_gain_fp": head["final"], "cos_fp": cos[:2048], "sin_fp": sin[:2048],
                               "layers": [layer] * LAYERS})
    return _keep("verifier", make)


def _blocks(r, out, nb, qtype):
    size = 144 if qtype == qk_gpu.Q4_K else 210
    raw = r.integers(0, 256, size=(out * nb, size), dtype=np.uint8)
    dv = r.uniform(0.0002, 0.001, size=out * nb).astype(np.float16).view(np.uint16)
    if qtype == qk_gpu.Q4_K:
        mv = r.uniform(0.0, 0.005, size=out * nb).astype(np.float16).view(np.uint16)
        raw[:, 0], raw[:, 1], raw[:, 2], raw[:, 3] = dv & 0xFF, dv >> 8, mv & 0xFF, mv >> 8
    else:
        raw[:, 208], raw[:, 209] = dv & 0xFF, dv >> 8
    return raw.reshape(-1)


def _experts():
    def make():
        r, out = np.random.default_rng(31), []
        for _ in range(EXPERTS):
            out.append(tuple(qk_gpu.register_weight(_blocks(r, o, n, q), o, n, q) for o, n, q in
                             ((NFF, ND // 256, qk_gpu.Q4_K), (NFF, ND // 256, qk_gpu.Q4_K),
                              (ND, NFF // 256, qk_gpu.Q6_K))))
        return out
    return _keep("experts", make)


def _nmc_layers(layers):
    def make():
        r, out = np.random.default_rng(32), []
        for n in range(layers):
            qkvo = [qk_gpu.register_weight(_blocks(r, o, i // 256, q), o, i // 256, q) for o, i, q in
                    ((NH * NHD, ND, qk_gpu.Q4_K), (NKV * NHD, ND, qk_gpu.Q4_K), (NKV * NHD, ND, qk_gpu.Q6_K),
                     (ND, NH * NHD, qk_gpu.Q4_K))]
            gain = qk_gpu.register_i64(r.integers(1 << 15, (1 << 17) + 1, size=(1, ND), dtype=np.int64))
            router = qk_gpu.register_i64(r.integers(-(1 << 20), 1 << 20, size=(EXPERTS, ND), dtype=np.int64))
            full = n % 4 == 3
            out.append(qk_gpu.ResidentMoeLayerSpec(n, gain, router, *qkvo, None if full else WINDOW, not full))
        return out
    return _keep(("nmc", layers), make)


# ---- one case: what a program has in hand, and one pass ---------------------------------------------------------------
def _ints(seed, shape, sigma, limit=None):
    """Normally distributed fixed-point values with standard deviation `sigma`, int64 on the GPU."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    v = torch.randn(shape, generator=gen, device="cuda", dtype=torch.float64) * sigma
    if limit is not None:
        v = v.clamp(-limit, limit)
    return v.round().to(torch.int64)


def _lens(case, seed):
    return np.random.default_rng(seed).integers(case["lo"], case["hi"] + 1, size=case["batch"]).astype(np.int64)


class _State(SimpleNamespace):
    """A case's inputs and handles; contexts are given back with it."""

    def __del__(self):
        for free in getattr(self, "frees", ()):
            free()


def _net(w, g, layers, batch, cap):
    return ResidentNet(B=batch, n_layers=layers, H=H, Hkv=HKV, hd=HD, d=D, dff=DFF, cap=cap, w=w, g=g, frac=FRAC,
                       page=64, kv32=True)


SAMPLER = SimpleNamespace(mode="top_p", temperature=0.6, top_k=20, top_p=0.95, min_p=0.0, seed=11, rep_penalty=0,
                          no_repeat_ngram=0)


def prepare(case, seed):
    kind = case["kind"]
    s = _State(kind=kind, lib=_lib.lib(), frees=[])
    rng = np.random.default_rng(seed)
    if kind == "linear":
        key = ("q1", case["out"], case["inp"], case["scale"])
        s.handle = _keep(key, lambda: _register(*_q1_host(case["out"], case["inp"], 300, case["scale"])))
        s.tokens = case["tokens"]
        s.x = _ints(seed, (case["tokens"], case["inp"]), 1 << FRAC)
        s.out = torch.empty((case["tokens"], case["out"]), dtype=torch.int64, device="cuda")
    elif kind == "monolith":
        s.w, s.g, _ = _model(case["layers"])
        s.dims = (case["tokens"], D, case["layers"], H, HKV, HD, DFF)
        s.x = _ints(seed, (case["tokens"], D), 1 << 12).cpu().numpy()
    elif kind == "ctx_step":
        w, g, _ = _model(case["layers"])
        s.pos = _lens(case, seed)
        s.ctx = gpu_native.decode_ctx_create((case["batch"], case["layers"], H, HKV, HD, D, DFF, VOCAB), w, g, FRAC, 1,
                                             INV_SQRT, int(case["hi"]) + 8)
        assert s.ctx is not None, _lib.last_error()
        s.frees.append(lambda h=s.ctx: gpu_native.decode_ctx_free(h))
        for b, n in enumerate(s.pos):
            kv = rng.integers(-(1 << 20), 1 << 20, size=(2, 1, HKV, int(n), HD), dtype=np.int64)
            kv = np.broadcast_to(kv, (2, case["layers"]) + kv.shape[2:])
            assert gpu_native.decode_ctx_seed_seq(s.ctx, b, kv[0], kv[1])
        s.x = _ints(seed, (case["batch"], D), 1 << 12).cpu().numpy()
    elif kind == "prefill":
        w, g, _ = _model(case["layers"])
        s.net = _net(w, g, case["layers"], 1, case["start"] + case["tokens"])
        s.frees.append(s.net.close)
        if case["start"]:
            s.net.fill_kv(seed, [case["start"]])
        s.start, s.tokens = case["start"], case["tokens"]
        s.x = _ints(seed, (case["tokens"], D), 1 << 12)
    elif kind == "generate":
        w, g, t = _model(case["layers"])
        s.ebits, s.escale, s.steps, s.mode = t["ebits"], t["escale"], case["steps"], case["mode"]
        s.lens = _lens(case, seed)
        s.net = _net(w, g, case["layers"], case["batch"], 64)
        s.frees.append(s.net.close)
        s.net.set_caps(s.lens + case["steps"] + 2)
        s.net.fill_kv(seed, s.lens)
        s.x0 = _ints(seed, (case["batch"], D), 1 << 12)
        s.x = torch.empty_like(s.x0)
        s.first = torch.from_numpy(rng.integers(0, VOCAB, size=case["batch"])).cuda()
        s.ids = torch.empty_like(s.first)
        s.logits = torch.empty((case["batch"], VOCAB), dtype=torch.int64, device="cuda")
        s.hist = torch.zeros((case["steps"], case["batch"]), dtype=torch.int64, device="cuda")
        s.rows = torch.zeros((case["batch"], 16 + case["steps"]), dtype=torch.int64, device="cuda")
        s.rows[:, :16] = torch.from_numpy(rng.integers(0, VOCAB, size=(case["batch"], 16))).cuda()
        s.rows_len = torch.empty(case["batch"], dtype=torch.int64, device="cuda")
    elif kind == "moe":
        e, m = _experts(), case["tokens"]
        pick = np.argsort(rng.random((m, EXPERTS)), axis=1)[:, :TOP].reshape(-1)
        s.handles = [(ctypes.c_int64 * (m * TOP))(*[e[i][k] for i in pick]) for k in range(3)]
        s.tokens = m
        s.h = _ints(seed, (m, ND), 1 << FRAC)
        s.gates = torch.from_numpy(rng.integers(1, 1 << FRAC, size=m * TOP)).cuda()
        s.out = torch.empty((m, ND), dtype=torch.int64, device="cuda")
    elif kind == "nmc_token":
        experts = _experts()
        cos, sin = _keep("nmc_tables", lambda: plain_tables(8192 + REPLY, NHD, 50000, FRAC))
        s.length, s.context, s.layers = case["context"] + REPLY, case["context"], case["layers"]
        s.specs = _nmc_layers(case["layers"])
        s.cache = qk_gpu.ResidentAttentionCache(case["layers"], s.length, ND, NH, NKV, NHD, FRAC,
                                                np.ascontiguousarray(cos[:s.length]),
                                                np.ascontiguousarray(sin[:s.length]))
        s.frees.append(s.cache.close)
        s.kv = rng.integers(-(1 << 20), 1 << 20, size=(2, NKV, s.context, NHD), dtype=np.int64)
        s.x = _ints(seed, (1, ND), 1 << 12).cpu().numpy()
        s.executor = qk_gpu.ResidentMoeTokenExecutor(
            s.cache, first_layer=0, layer_count=case["layers"], n_experts=EXPERTS, n_used=TOP, d_model=ND,
            expert_ffn=NFF, fw=FW, eps=1, lookup_expert=lambda l, i: experts[i], load_expert=lambda l, i: experts[i])
        for n in range(s.layers):
            s.cache.import_layer(n, s.kv[0], s.kv[1])
        s.executor.prepare(s.specs)
    else:
        s.model = _verifier()
        s.ids = [int(v) for v in rng.integers(0, VOCAB, size=case["tokens"])]
        s.out = case["out"]
    return s


def run(s):
    if s.kind == "linear":
        st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
        rc = s.lib.imie_q1_apply_dev(s.handle, ctypes.c_void_p(s.x.data_ptr()), s.tokens, FRAC,
                                     ctypes.c_void_p(s.out.data_ptr()), st)
        assert rc == 0, _lib.last_error()
        return s.out
    if s.kind == "monolith":
        logits, k, v = gpu_native.prefill_forward_gpu(s.x, s.dims, s.w, s.g, FRAC, 1, INV_SQRT, export_kv=True)
        assert logits is not None, _lib.last_error()
        return logits, k, v
    if s.kind == "ctx_step":
        logits = gpu_native.decode_step(s.ctx, s.x, s.pos, VOCAB)
        assert logits is not None, _lib.last_error()
        return logits
    if s.kind == "prefill":
        with torch.cuda.stream(s.net.stream):
            x = s.x.clone()      # the layers update it in place
        status = s.net.forward(x, [s.start], s.tokens)
        assert status == 0
        return x
    if s.kind == "generate":
        with torch.cuda.stream(s.net.stream):
            s.x.copy_(s.x0)
            s.ids.copy_(s.first)
            if s.mode != "greedy":
                s.rows_len.fill_(16)
        status = s.net.forward(s.x, s.lens, 1)
        assert status == 0
        if s.mode == "greedy":
            logits, tokens = s.net.decode(s.ebits, s.escale, s.ids, s.steps, hist=s.hist, logits=s.logits)
        else:
            logits = s.net.decode_sampled(s.ebits, s.escale, s.ids, s.steps, SAMPLER, FRAC, s.rows, s.rows_len,
                                          logits=s.logits)
            tokens = s.rows
        with torch.cuda.stream(s.net.stream):
            tokens = tokens.cpu()        # the program reads the text
        return s.x, logits, tokens
    if s.kind == "moe":
        st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
        rc = s.lib.imie_moe_ffn_batched_dev(*s.handles, s.tokens, TOP, ctypes.c_void_p(s.h.data_ptr()),
                                            ctypes.c_void_p(s.gates.data_ptr()), ND, NFF, FRAC, FW,
                                            ctypes.c_void_p(s.out.data_ptr()), st)
        assert rc == 0, _lib.last_error()
        return s.out
    if s.kind == "nmc_token":
        if s.cache.length(0) >= s.length:        # this reply is full: the next request's prompt
            s.cache.reset()
            for n in range(s.layers):
                s.cache.import_layer(n, s.kv[0], s.kv[1])
        return s.executor.run(s.x, s.specs)
    model = s.model
    full = model.logits_dev(s.ids)
    at = list(range(len(s.ids) - s.out - 1, len(s.ids) - 1))
    rows = model.take_rows(full, at)
    tokens = model.select(rows, SAMPLER, [n + 1 for n in at], [s.ids[:n + 1] for n in at])
    digests = np.stack([np.frombuffer(bytes.fromhex(d), dtype=np.uint8) for d in model.digests(rows)])
    return full, np.array(tokens, dtype=np.int64), digests


# ---- what a pass cannot do without --------------------------------------------------------------------------------------
def _linear_work(tokens, out, inp, scale_bytes=4):
    """A Q1_0 projection: its bits and scales once, activations in and out once."""
    return out * inp // 8 + out * (inp // 128) * scale_bytes + tokens * (out + inp) * 8, 2 * tokens * out * inp


def _layers_work(layers, keys, visible, rows):
    """`layers` 8B layers over `rows` new rows: weights once, the cache that is seen once at 4 bytes an element."""
    weights = LAYER_WEIGHTS // 8 + LAYER_WEIGHTS // 128 * 4
    nbytes = layers * (weights + keys * 2 * HKV * HD * 4) + 2 * rows * D * 8
    return nbytes, layers * (2 * rows * LAYER_WEIGHTS + 4 * visible * H * HD)


def work(case):
    kind = case["kind"]
    head_b, head_f = _linear_work(1, VOCAB, D)
    if kind == "linear":
        b, f = _linear_work(case["tokens"], case["out"], case["inp"], 4 if case["scale"] == "i32" else 8)
    elif kind == "monolith":
        t = case["tokens"]
        b, f = _layers_work(case["layers"], t, t * (t + 1) // 2, t)
        b, f = b + head_b + case["layers"] * 2 * HKV * t * HD * 8, f + head_f
    elif kind == "ctx_step":
        keys = case["batch"] * (case["lo"] + case["hi"]) // 2
        b, f = _layers_work(case["layers"], 2 * keys, keys, case["batch"])      # an int64 cache: 8 bytes an element
        b, f = b + head_b + (case["batch"] - 1) * VOCAB * 8, f + case["batch"] * head_f
    elif kind == "prefill":
        t, n = case["tokens"], case["start"]
        b, f = _layers_work(case["layers"], n + t, t * n + t * (t + 1) // 2, t)
    elif kind == "generate":
        keys = case["batch"] * (case["lo"] + case["hi"]) // 2
        b, f = _layers_work(case["layers"], keys, keys, case["batch"])
        b, f = (case["steps"] + 1) * b, (case["steps"] + 1) * f
        b += case["steps"] * (head_b + (case["batch"] - 1) * VOCAB * 8)
        f += case["steps"] * case["batch"] * head_f
    elif kind == "moe":
        m = case["tokens"]
        used = EXPERTS * (1 - (1 - TOP / EXPERTS) ** m)
        b, f = used * EXPERT_BYTES + 2 * m * ND * 8, 2 * m * TOP * 3 * ND * NFF
    elif kind == "nmc_token":
        qkvo = (NH * NHD + NKV * NHD) * (ND // 256) * 144 + NKV * NHD * (ND // 256) * 210 + ND * (NH * NHD // 256) * 144
        keys = sum(case["context"] if n % 4 == 3 else min(case["context"], WINDOW) for n in range(case["layers"]))
        b = case["layers"] * (qkvo + EXPERTS * ND * 8 + TOP * EXPERT_BYTES) + keys * 2 * NKV * NHD * 8
        f = case["layers"] * 2 * (2 * NH * NHD * ND + 2 * NKV * NHD * ND + EXPERTS * ND + TOP * 3 * ND * NFF)
        f += 4 * keys * NH * NHD
    else:
        t = case["tokens"]
        b, f = _layers_work(LAYERS, t, t * (t + 1) // 2, t)
        b, f = b + head_b + (t + case["out"]) * VOCAB * 8, f + t * head_f
    return {"bytes": float(b), "flops": float(f)}


def tolerance(case):
    return "exact"


def exact(case, seed):
    """The linear in 64-bit whole numbers. The other calls chain dozens of such rounded steps, whole numbers all of
    them, which have to be the same to the bit."""
    if case["kind"] != "linear":
        return None
    bits, scale = _q1_host(case["out"], case["inp"], 300, case["scale"])
    x = _ints(seed, (case["tokens"], case["inp"]), 1 << FRAC).cpu().numpy()
    out = np.zeros((case["tokens"], case["out"]), dtype=np.int64)
    with np.errstate(over="ignore"):
        for b in range(case["inp"] // 128):
            sign = np.unpackbits(bits[:, b], axis=1, bitorder="little").astype(np.float64) * 2 - 1
            total = np.rint(x[:, b * 128:(b + 1) * 128].astype(np.float64) @ sign.T).astype(np.int64)
            out += (total * scale[None, :, b]) >> FRAC
    return out
