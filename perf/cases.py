"""The calls a user of this library makes, with the sizes they make them at, for timing and for
comparing outputs.

Four kinds of case, after the entry points of models_amd.attention:

* ``host``     one decode layer-step through the host-buffer call, as the Java forward pass makes
               it when its projections run on the CPU;
* ``token``    one decode token through every layer of a model (one device call per layer);
* ``sessions`` one decode layer-step of many sessions of different lengths in one call;
* ``prefill``  RoPE, cache append and causal attention of one layer's prompt or prompt chunk;
* ``project``  the GGUF-quantized projections around attention;
* ``block``    a prompt through one layer's whole attention block: Q/K/V projection, prefill,
               output projection and residual.

Model shapes are the ones the tests and the benchmark of this repository use (query heads, KV
heads, head dimension, RoPE kind and base, window, QK-norm).
"""

import math

import numpy as np
import torch

from models_amd import attention as A

# name: (query heads, KV heads, head dim, NeoX pairs, RoPE base, f16 cache, QK-norm)
MODELS = {
    "llama-1b": (32, 8, 64, False, 5e5, True, False),
    "llama-3b": (24, 8, 128, False, 5e5, True, False),
    "qwen2.5-1.5b": (12, 2, 128, True, 1e6, True, False),
    "qwen3-0.6b": (16, 8, 128, True, 1e6, False, True),
    "gemma3-1b": (4, 1, 256, True, 1e6, True, True),
    "gemma4-full": (8, 1, 512, True, 1e6, True, True),
}
EPS = 1e-6

FORMATS = {"q4_0": (A.WEIGHTS_Q4_0,), "q8_0": (A.WEIGHTS_Q8_0,), "q5_0": (A.WEIGHTS_Q5_0,),
           "q4_k": (A.WEIGHTS_Q4_K,), "q6_k": (A.WEIGHTS_Q6_K,),
           # a Q4_K_M file's Q, K and V
           "q4_k_m": (A.WEIGHTS_Q4_K, A.WEIGHTS_Q4_K, A.WEIGHTS_Q6_K)}


def listed():
    return [
        # The smallest call: one layer of one token at a short context, f32 cache, host buffers.
        {"name": "decode_host_512", "kind": "host", "model": "qwen3-0.6b", "position": 512},
        # Interactive generation at a 4k context: a token through a 16-layer model.
        {"name": "token_4k", "kind": "token", "model": "llama-1b", "layers": 16, "position": 4100,
         "window": 0, "pattern": 0},
        # Long-context generation: 26 layers, five sliding-window layers to each global one.
        {"name": "token_32k_sliding", "kind": "token", "model": "gemma3-1b", "layers": 26,
         "position": 32704, "window": 512, "pattern": 6},
        # A serving batch: 64 sessions of 256 to 16384 positions, one layer, one call.
        {"name": "sessions_64_ragged", "kind": "sessions", "model": "qwen2.5-1.5b", "sessions": 64,
         "low": 256, "high": 16384},
        # A chat-sized prompt (odd length) on a small model: few workgroups, launch-bound.
        {"name": "prefill_77", "kind": "prefill", "model": "llama-1b", "start": 0, "rows": 77,
         "window": 0},
        # The 2k-token prompt the benchmark quotes, f16 cache.
        {"name": "prefill_2k", "kind": "prefill", "model": "llama-3b", "start": 0, "rows": 2048,
         "window": 0},
        # A chunk of a long prompt in a sliding-window layer, head dim 256, QK-norm.
        {"name": "prefill_chunk_window", "kind": "prefill", "model": "gemma3-1b", "start": 3001,
         "rows": 1000, "window": 512},
        # A 1000-token prompt on an f32 cache with QK-norm.
        {"name": "prefill_f32_1000", "kind": "prefill", "model": "qwen3-0.6b", "start": 0,
         "rows": 1000, "window": 0},
        # Q/K/V of one decode token, Q4_0.
        {"name": "project_token_q4_0", "kind": "project", "format": "q4_0", "batch": 1,
         "cols": 2048, "q_rows": 2048, "kv_rows": 512, "residual": False},
        # The output projection of a chat-sized prompt with the residual added in place, Q8_0.
        {"name": "project_77_q8_0", "kind": "project", "format": "q8_0", "batch": 77,
         "cols": 2048, "q_rows": 2048, "kv_rows": 0, "residual": True},
        # Q/K/V of a 2k-token prompt from a Q4_K_M file (Q4_K, Q4_K, Q6_K).
        {"name": "project_2k_q4_k_m", "kind": "project", "format": "q4_k_m", "batch": 2048,
         "cols": 3072, "q_rows": 3072, "kv_rows": 1024, "residual": False},
        # A whole attention block on a 1000-token prompt, Q4_0 weights.
        {"name": "block_1000_q4_0", "kind": "block", "model": "llama-3b", "format": "q4_0",
         "rows": 1000, "dim": 3072},
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(("host", "token", "sessions", "prefill", "prefill", "project", "project", "block"))
    if kind == "host":
        return {"kind": kind, "model": rng.choice(sorted(MODELS)), "position": _log_int(rng, 16, 8192)}
    if kind == "token":
        model = rng.choice(sorted(MODELS))
        sliding = model.startswith("gemma")
        return {"kind": kind, "model": model, "layers": rng.randint(1, 20),
                "position": _log_int(rng, 100, 16384), "window": 512 if sliding else 0,
                "pattern": 6 if sliding else 0}
    if kind == "sessions":
        high = _log_int(rng, 300, 12000)
        return {"kind": kind, "model": rng.choice(("llama-1b", "llama-3b", "qwen2.5-1.5b", "gemma3-1b")),
                "sessions": rng.randint(2, 48), "low": rng.randint(1, high // 2), "high": high}
    if kind == "prefill":
        model = rng.choice(sorted(MODELS))
        return {"kind": kind, "model": model, "start": rng.choice((0, 0, _log_int(rng, 1, 4000))),
                "rows": _log_int(rng, 2, 2048),
                "window": 512 if model == "gemma3-1b" and rng.random() < 0.7 else 0}
    if kind == "project":
        fmt = rng.choice(sorted(FORMATS))
        residual = rng.random() < 0.4
        return {"kind": kind, "format": fmt, "batch": _log_int(rng, 1, 2048),
                "cols": 256 * rng.randint(4, 12), "q_rows": rng.randint(500, 3072),
                "kv_rows": 0 if residual else rng.randint(100, 1024), "residual": residual}
    return {"kind": kind, "model": rng.choice(("llama-1b", "llama-3b", "qwen2.5-1.5b")),
            "format": rng.choice(("q4_0", "q8_0", "q4_k", "q4_k_m")), "rows": _log_int(rng, 16, 1000),
            "dim": 256 * rng.randint(6, 12)}


# ---------------------------------------------------------------- the program around the calls

_program = {}


def _library():
    """One library context, as a program holds it."""
    if "lib" not in _program:
        _program["lib"] = A.HipAttentionLibrary(0)
    return _program["lib"]


def _rope(dim, theta, positions):
    """A model's RoPE table, kept for as long as the program runs."""
    positions = -(-positions // 4096) * 4096
    key = ("rope", dim, theta, positions)
    if key not in _program:
        _program[key] = _library().rotary_table(dim, theta, 1.0, max_positions=positions)
    return _program[key]


class State:
    """Inputs, outputs and handles of one case; its cache is closed with it."""

    def __init__(self, **fields):
        self.__dict__.update(fields)

    def __del__(self):
        for name in ("kv", "norm"):
            handle = self.__dict__.get(name)
            if handle is not None:
                handle.close()


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _randn(g, *shape):
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32)


def _norm_weights(g, d):
    return 1.0 + 0.1 * _randn(g, d), 1.0 + 0.1 * _randn(g, d)


def _is_global(case, layer):
    return case["pattern"] == 0 or layer % case["pattern"] == case["pattern"] - 1


def _layer_window(case, layer):
    return 0 if _is_global(case, layer) else case["window"]


def _decode_calls(layers, q, k, v, out):
    """Per layer: its parameters and the (pointer, elements) pairs of its rows of q, k, v and out."""
    calls = []
    for i, layer in enumerate(layers):
        buffers = []
        for t in (q, k, v, out):
            rows = t.reshape(len(layers), -1)[i]
            buffers += [rows.data_ptr(), rows.numel()]
        calls.append((layer, buffers))
    return calls


def _fill(lib, kv, layer, keys, values, first, sequence=0):
    """Caches rotated keys and values of positions first .. of one session."""
    n = keys.shape[0]
    store = A.AttentionLayer(layer.layer, kv.num_kv_heads, layer.sliding_window, layer.neox,
                             rope=layer.rope, qk_norm=layer.qk_norm)
    kv.append_device(store, np.full(n, sequence, np.uint32), np.arange(first, first + n, dtype=np.uint32),
                     keys.data_ptr(), keys.numel(), keys.data_ptr(), keys.numel(),
                     values.data_ptr(), values.numel())
    lib.synchronize()


def _model_norm(lib, model, g):
    """(norm handle or None, q weight, k weight) of a model's layers."""
    d = MODELS[model][2]
    if not MODELS[model][6]:
        return None, None, None
    wq, wk = _norm_weights(g, d)
    return lib.qk_norm(d, wq.cpu().numpy(), wk.cpu().numpy(), EPS), wq, wk


# ---- inputs, from the seed alone (prepare and exact draw the same ones in the same order)

def _session_lengths(case, seed):
    r = np.random.RandomState(seed % (1 << 31))
    return r.randint(case["low"], case["high"] + 1, case["sessions"])


def _token_layers(case):
    """Per layer of a token case: (window, first cached position that is ever visible)."""
    for layer in range(case["layers"]):
        w = _layer_window(case, layer)
        yield layer, w, max(0, case["position"] - w + 1) // 32 * 32 if w else 0


def _quantize(w, fmt):
    """GGUF blocks of a [rows, cols] float weight matrix (uint8 on the GPU), and in float64 the
    values they stand for."""
    rows, cols = w.shape

    def f16_bytes(x):
        return x.to(torch.float16).contiguous().view(torch.uint8).reshape(*x.shape, 2)

    if fmt in (A.WEIGHTS_Q4_0, A.WEIGHTS_Q8_0, A.WEIGHTS_Q5_0):
        x = w.reshape(rows, cols // 32, 32)
        if fmt == A.WEIGHTS_Q8_0:
            d = (x.abs().amax(-1) / 127).to(torch.float16)
            q = torch.round(x / d.float().clamp_min(1e-8)[..., None]).clamp(-127, 127)
            body = q.to(torch.int8).contiguous().view(torch.uint8)
        else:
            half = 8 if fmt == A.WEIGHTS_Q4_0 else 16
            at = x.abs().argmax(-1, keepdim=True)
            d = (x.gather(-1, at)[..., 0] / -half).to(torch.float16)
            dd = d.float()
            dd = torch.where(dd == 0, torch.ones_like(dd), dd)
            u = (torch.round(x / dd[..., None]) + half).clamp(0, 2 * half - 1).to(torch.int32)
            q = (u - half).float()
            body = ((u[..., :16] & 15) | ((u[..., 16:] & 15) << 4)).to(torch.uint8)
            if half == 16:
                high = ((u >> 4).reshape(rows, cols // 32, 4, 8)
                        << torch.arange(8, device=w.device)).sum(-1).to(torch.uint8)
                body = torch.cat([high, body], -1)
        blocks = torch.cat([f16_bytes(d), body], -1)
        return blocks.reshape(-1).contiguous(), (d.double()[..., None] * q.double()).reshape(rows, cols)

    n = cols // 256
    if fmt == A.WEIGHTS_Q4_K:
        x = w.reshape(rows, n, 8, 32)
        low = (-x.amin(-1)).clamp_min(0)
        step = (x.amax(-1) + low) / 15
        d, dmin = ((v.amax(-1) / 63).to(torch.float16) for v in (step, low))
        sc = torch.round(step / d.float().clamp_min(1e-8)[..., None]).clamp(0, 63).to(torch.int32)
        mn = torch.round(low / dmin.float().clamp_min(1e-8)[..., None]).clamp(0, 63).to(torch.int32)
        scale, offset = d.float()[..., None] * sc, dmin.float()[..., None] * mn
        u = torch.round((x + offset[..., None]) / scale.clamp_min(1e-8)[..., None]).clamp(0, 15).to(torch.int32)
        packed = torch.cat([(sc[..., :4] & 63) | ((sc[..., 4:] >> 4) << 6),
                            (mn[..., :4] & 63) | ((mn[..., 4:] >> 4) << 6),
                            (sc[..., 4:] & 15) | ((mn[..., 4:] & 15) << 4)], -1).to(torch.uint8)
        body = (u[..., 0::2, :] | (u[..., 1::2, :] << 4)).to(torch.uint8).reshape(rows, n, 128)
        blocks = torch.cat([f16_bytes(d), f16_bytes(dmin), packed, body], -1)
        value = (d.double()[..., None] * sc)[..., None] * u - (dmin.double()[..., None] * mn)[..., None]
        return blocks.reshape(-1).contiguous(), value.reshape(rows, cols)

    x = w.reshape(rows, n, 16, 16)  # Q6_K
    step = x.gather(-1, x.abs().argmax(-1, keepdim=True))[..., 0] / -32
    d = (step.abs().amax(-1) / 127).to(torch.float16)
    sc = torch.round(step / d.float().clamp_min(1e-8)[..., None]).clamp(-127, 127).to(torch.int32)
    scale = d.float()[..., None] * sc
    scale = torch.where(scale == 0, torch.ones_like(scale), scale)
    u = (torch.round(x / scale[..., None]) + 32).clamp(0, 63).to(torch.int32)
    run = u.reshape(rows, n, 2, 4, 32)  # two halves of four 32-element runs
    low = torch.stack([(run[..., 0, :] & 15) | ((run[..., 2, :] & 15) << 4),
                       (run[..., 1, :] & 15) | ((run[..., 3, :] & 15) << 4)], -2)
    high = sum((run[..., i, :] >> 4) << (2 * i) for i in range(4))
    blocks = torch.cat([low.to(torch.uint8).reshape(rows, n, 128), high.to(torch.uint8).reshape(rows, n, 64),
                        sc.to(torch.int8).contiguous().view(torch.uint8), f16_bytes(d)], -1)
    value = (d.double()[..., None] * sc)[..., None] * (u - 32)
    return blocks.reshape(-1).contiguous(), value.reshape(rows, cols)


def _weights(g, fmt, rows, cols):
    return _quantize(_randn(g, rows, cols) * (1.0 / math.sqrt(cols)), fmt)


def _project_inputs(case, seed):
    """(activations, [(format, rows, blocks, float64 values)], residual or None)."""
    g = _gen(seed)
    rows = [case["q_rows"]] + ([case["kv_rows"]] * 2 if case["kv_rows"] else [])
    formats = FORMATS[case["format"]]
    mats = [(f, r) + _weights(g, f, r, case["cols"])
            for f, r in ((formats[min(i, len(formats) - 1)], r) for i, r in enumerate(rows))]
    x = _randn(g, case["batch"], case["cols"])
    residual = _randn(g, case["batch"], rows[0]) if case["residual"] else None
    return x, mats, residual


def _block_inputs(case, seed):
    """(hidden state, its normed form, Q/K/V matrices, output matrix), as _project_inputs."""
    hq, hkv, d = MODELS[case["model"]][:3]
    g = _gen(seed)
    formats = FORMATS[case["format"]]
    qkv = [(f, r) + _weights(g, f, r, case["dim"])
           for f, r in ((formats[min(i, len(formats) - 1)], r)
                        for i, r in enumerate((hq * d, hkv * d, hkv * d)))]
    out = (formats[0], case["dim"]) + _weights(g, formats[0], case["dim"], hq * d)
    x = _randn(g, case["rows"], case["dim"])
    return x, x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS), qkv, out


def _grouped(lib, mats, x, out):
    batch, cols = x.shape
    lib.quantized_grouped_matmul_device([m[0] for m in mats], [m[2].data_ptr() for m in mats],
                                        [m[2].numel() for m in mats], [m[1] for m in mats],
                                        x.data_ptr(), x.numel(), out.data_ptr(), out.numel(), batch, cols)


# ---------------------------------------------------------------- prepare

def prepare(case, seed):
    state = _prepare(case, seed)
    torch.cuda.synchronize()
    return state


def _prepare(case, seed):
    lib, kind = _library(), case["kind"]
    if kind == "project":
        x, mats, residual = _project_inputs(case, seed)
        mats = [m[:3] for m in mats]
        out = torch.empty(x.shape[0] * sum(m[1] for m in mats), device="cuda")
        return State(kind=kind, lib=lib, x=x, mats=mats, residual=residual, out=out)
    hq, hkv, d, neox, theta, half, _ = MODELS[case["model"]]
    if kind == "block":
        x, xn, qkv, wo = _block_inputs(case, seed)
        n, dim = x.shape
        kv = lib.kv_cache(1, n, hkv, d, d, half_precision=half)
        layer = A.AttentionLayer(0, hq, neox=neox, rope=_rope(d, theta, n))
        return State(kind=kind, lib=lib, kv=kv, layer=layer, x=x, xn=xn, qkv=[m[:3] for m in qkv], wo=wo[:3],
                     proj=torch.empty(n * (hq + 2 * hkv) * d, device="cuda"),
                     attn=torch.empty(n, hq * d, device="cuda"), out=torch.empty(n, dim, device="cuda"))

    g = _gen(seed)
    norm, _, _ = _model_norm(lib, case["model"], g)
    if kind in ("host", "token"):
        token = case if kind == "token" else dict(case, layers=1, window=0, pattern=0)
        pos = token["position"]
        rope = _rope(d, theta, pos + 1)
        # A sliding layer keeps its window in a ring; a global one keeps every position.
        specs = [A.LayerSpec(hkv, d, d, w + 32 if w else 0) for _, w, _ in _token_layers(token)]
        kv = lib.layered_kv_cache(specs, pos + 1, half_precision=half)
        layers = []
        for i, w, first in _token_layers(token):
            layer = A.AttentionLayer(i, hq, w, neox, rope=rope, qk_norm=norm)
            k, v = _randn(g, pos - first, hkv * d), _randn(g, pos - first, hkv * d)
            torch.cuda.synchronize()
            _fill(lib, kv, layer, k, v, first)
            layers.append(layer)
        q, k, v = (_randn(g, len(layers), h * d) for h in (hq, hkv, hkv))
        if kind == "host":
            return State(kind=kind, kv=kv, norm=norm, layer=layers[0], position=[pos],
                         q=q.cpu().numpy(), k=k.cpu().numpy(), v=v.cpu().numpy())
        out = torch.empty(len(layers), hq * d, device="cuda")
        return State(kind=kind, kv=kv, norm=norm, sequences=np.zeros(1, np.uint32),
                     positions=np.full(1, pos, np.uint32), q=q, k=k, v=v, out=out,
                     calls=_decode_calls(layers, q, k, v, out))
    if kind == "sessions":
        lengths = _session_lengths(case, seed)
        rope = _rope(d, theta, case["high"] + 1)
        kv = lib.kv_cache(1, case["high"] + 1, hkv, d, d, half_precision=half, sequences=len(lengths))
        layer = A.AttentionLayer(0, hq, neox=neox, rope=rope, qk_norm=norm)
        for s, n in enumerate(lengths):
            k, v = _randn(g, int(n), hkv * d), _randn(g, int(n), hkv * d)
            torch.cuda.synchronize()
            _fill(lib, kv, layer, k, v, 0, s)
        q, k, v = (_randn(g, len(lengths), h * d) for h in (hq, hkv, hkv))
        out = torch.empty(len(lengths), hq * d, device="cuda")
        return State(kind=kind, kv=kv, norm=norm, sequences=np.arange(len(lengths), dtype=np.uint32),
                     positions=lengths.astype(np.uint32), q=q, k=k, v=v, out=out,
                     calls=_decode_calls([layer], q, k, v, out))
    start, n, w = case["start"], case["rows"], case["window"]
    kv = lib.kv_cache(1, start + n, hkv, d, d, half_precision=half)
    layer = A.AttentionLayer(0, hq, w, neox, rope=_rope(d, theta, start + n), qk_norm=norm)
    if start:
        k, v = _randn(g, start, hkv * d), _randn(g, start, hkv * d)
        torch.cuda.synchronize()
        _fill(lib, kv, layer, k, v, 0)
    q, k, v = (_randn(g, n, h * d) for h in (hq, hkv, hkv))
    return State(kind=kind, kv=kv, norm=norm, layer=layer, start=start, q=q, k=k, v=v,
                 out=torch.empty(n, hq * d, device="cuda"))


# ---------------------------------------------------------------- run

def run(s):
    if s.kind == "host":
        return s.kv.decode(s.layer, s.position, s.q, s.k, s.v)
    if s.kind in ("token", "sessions"):
        for layer, buffers in s.calls:
            s.kv.decode_device(layer, s.sequences, s.positions, *buffers)
        return s.out
    if s.kind == "prefill":
        s.kv.prefill_device(s.layer, 0, s.start, s.q.shape[0], s.q.data_ptr(), s.q.numel(), s.k.data_ptr(),
                            s.k.numel(), s.v.data_ptr(), s.v.numel(), s.out.data_ptr(), s.out.numel())
        return s.out
    if s.kind == "project":
        batch, cols = s.x.shape
        if s.residual is not None:
            fmt, rows, blocks = s.mats[0]
            s.lib.quantized_matmul_device(fmt, blocks.data_ptr(), blocks.numel(), s.x.data_ptr(),
                                          s.x.numel(), s.out.data_ptr(), s.out.numel(), batch, rows, cols,
                                          s.residual.data_ptr(), A.ADDEND_RESIDUAL)
        else:
            _grouped(s.lib, s.mats, s.x, s.out)
        return s.out
    n = s.x.shape[0]
    _grouped(s.lib, s.qkv, s.xn, s.proj)
    q, k, v = s.proj.split([n * m[1] for m in s.qkv])
    s.kv.prefill_device(s.layer, 0, 0, n, q.data_ptr(), q.numel(), k.data_ptr(), k.numel(), v.data_ptr(),
                        v.numel(), s.attn.data_ptr(), s.attn.numel())
    fmt, rows, blocks = s.wo
    s.lib.quantized_matmul_device(fmt, blocks.data_ptr(), blocks.numel(), s.attn.data_ptr(), s.attn.numel(),
                                  s.out.data_ptr(), s.out.numel(), n, rows, s.attn.shape[1], s.x.data_ptr(),
                                  A.ADDEND_RESIDUAL)
    return s.out, s.attn


# ---------------------------------------------------------------- work and tolerance

_BLOCK_BYTES = {A.WEIGHTS_Q4_0: 18 / 32, A.WEIGHTS_Q8_0: 34 / 32, A.WEIGHTS_Q5_0: 22 / 32,
                A.WEIGHTS_Q4_K: 144 / 256, A.WEIGHTS_Q6_K: 210 / 256}


def _attention_work(model, visible, rows, cached):
    """`visible`: (query, key) pairs per query head; `cached`: cache rows read; `rows`: new rows."""
    hq, hkv, d, _, _, half, _ = MODELS[model]
    e = 2 if half else 4
    return {"flops": 4.0 * hq * d * visible,
            "bytes": 2.0 * hkv * d * e * (cached + rows) + 4.0 * rows * d * (2 * hq + 2 * hkv)}


def _project_work(formats, sizes, batch, cols, residual):
    rows = sum(sizes)
    weights = sum(r * cols * _BLOCK_BYTES[formats[min(i, len(formats) - 1)]] for i, r in enumerate(sizes))
    return {"flops": 2.0 * batch * rows * cols,
            "bytes": weights + 4.0 * batch * (cols + rows * (2 if residual else 1))}


def _sum(parts):
    return {key: sum(p[key] for p in parts) for key in ("bytes", "flops")}


def _causal_pairs(start, n, window):
    seen = np.arange(start, start + n) + 1
    return float(np.minimum(seen, window).sum() if window else seen.sum())


def work(case):
    kind = case["kind"]
    if kind == "host":
        return _attention_work(case["model"], case["position"] + 1, 1, case["position"])
    if kind == "token":
        seen = [min(case["position"] + 1, w) if w else case["position"] + 1 for _, w, _ in _token_layers(case)]
        return _sum([_attention_work(case["model"], s, 1, s - 1) for s in seen])
    if kind == "sessions":
        mean = 0.5 * (case["low"] + case["high"]) * case["sessions"]
        return _attention_work(case["model"], mean + case["sessions"], case["sessions"], mean)
    if kind == "prefill":
        w = case["window"]
        cached = min(case["start"], w - 1) if w else case["start"]
        return _attention_work(case["model"], _causal_pairs(case["start"], case["rows"], w), case["rows"], cached)
    if kind == "project":
        sizes = [case["q_rows"]] + ([case["kv_rows"]] * 2 if case["kv_rows"] else [])
        return _project_work(FORMATS[case["format"]], sizes, case["batch"], case["cols"], case["residual"])
    hq, hkv, d = MODELS[case["model"]][:3]
    formats, n = FORMATS[case["format"]], case["rows"]
    return _sum([_project_work(formats, (hq * d, hkv * d, hkv * d), n, case["dim"], False),
                 _attention_work(case["model"], _causal_pairs(0, n, 0), n, 0),
                 _project_work(formats[:1], (case["dim"],), n, hq * d, True)])


def tolerance(case):
    kind = case["kind"]
    if kind == "project":
        return {"rel": 2e-6, "max": 1e-4}  # float32 chains over the blocks, integer dots exact
    if kind == "block":
        return {"rel": 2.5e-3, "max": 0.1}  # float16 attention, then Q8 activations that round it again
    if kind == "prefill" and MODELS[case["model"]][5]:
        return {"rel": 1.5e-3, "max": 0.1}  # float16 queries and probabilities
    return {"rel": 1e-5, "max": 1e-3}     # float32 products (an f16 cache only rounds what it stores)


# ---------------------------------------------------------------- the same in 64 bits

def _rotate(x, positions, theta, neox):
    """RoPE of x [rows, heads, d] (float64) at `positions`: float32 angles, as the model defines them."""
    d = x.shape[-1]
    freq = torch.tensor([1.0 / theta ** (2 * i / d) for i in range(d // 2)], dtype=torch.float64).float().cuda()
    angle = (positions.float()[:, None] * freq).double()
    c, s = (f(angle).float().double()[:, None, :] for f in (torch.cos, torch.sin))
    y = torch.empty_like(x)
    a, b = (slice(0, d // 2), slice(d // 2, d)) if neox else (slice(0, d, 2), slice(1, d, 2))
    y[..., a] = x[..., a] * c - x[..., b] * s
    y[..., b] = x[..., a] * s + x[..., b] * c
    return y


def _heads(x, d, weight, positions, theta, neox):
    """Rows [n, heads * d] normalised and rotated per head, in 64 bits."""
    x = x.double().reshape(x.shape[0], -1, d)
    if weight is not None:
        x = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * weight.double()
    return _rotate(x, positions, theta, neox)


def _attend(model, q, k, v, first_q, first_k, window, wq, wk):
    """Causal attention of raw rows q (positions first_q ..) over raw k, v (first_k ..)."""
    hq, hkv, d, neox, theta, half, _ = MODELS[model]
    n, m = q.shape[0], k.shape[0]
    pq = torch.arange(first_q, first_q + n, device="cuda")
    pk = torch.arange(first_k, first_k + m, device="cuda")
    qs = _heads(q, d, wq, pq, theta, neox)
    ks = _heads(k, d, wk, pk, theta, neox)
    vs = v.double().reshape(m, hkv, d)
    if half:
        ks, vs = ks.float().half().double(), vs.half().double()
    hidden = pk[None, :] > pq[:, None]
    if window:
        hidden = hidden | (pk[None, :] <= pq[:, None] - window)
    out = torch.empty(n, hq, d, dtype=torch.float64, device="cuda")
    for h in range(hq):
        scores = (qs[:, h] @ ks[:, h * hkv // hq].T.contiguous()) / math.sqrt(d)
        out[:, h] = torch.softmax(scores.masked_fill(hidden, -math.inf), -1) @ vs[:, h * hkv // hq]
    return out.reshape(n, hq * d)


def _over(number, x):
    """number / x rounded once (a scalar over a tensor may go by a rounded reciprocal), 0 where x is 0."""
    return torch.where(x == 0, torch.zeros_like(x), torch.div(torch.full_like(x, number), x))


def _activations(x, kquant):
    """What the Q8_0 or Q8_K activation blocks of x stand for, in 64 bits."""
    if kquant:
        b = x.reshape(x.shape[0], -1, 256)
        top = b.gather(-1, b.abs().argmax(-1, keepdim=True))
        inverse = _over(-127.0, top)
        q = torch.round(inverse * b).clamp(max=127)
        scale = _over(1.0, inverse)
    else:
        b = x.reshape(x.shape[0], -1, 32)
        top = b.abs().amax(-1, keepdim=True)
        q = torch.round(b * _over(127.0, top))
        scale = torch.div(top, torch.full_like(top, 127.0)).half()
    return (scale.double() * q.double()).reshape(x.shape)


def _products(x, mats):
    kquant = mats[0][0] in (A.WEIGHTS_Q4_K, A.WEIGHTS_Q6_K)
    xq = _activations(x, kquant)
    return [xq @ m[3].T.contiguous() for m in mats]


def exact(case, seed):
    kind = case["kind"]
    if kind == "project":
        x, mats, residual = _project_inputs(case, seed)
        got = _products(x, mats)
        if residual is not None:
            got[0] = got[0] + residual.double()
        return torch.cat([y.reshape(-1) for y in got])
    model = case["model"]
    hq, hkv, d = MODELS[model][:3]
    if kind == "block":
        x, xn, qkv, wo = _block_inputs(case, seed)
        q, k, v = (y.float() for y in _products(xn, qkv))
        attn = _attend(model, q, k, v, 0, 0, 0, None, None)
        return _products(attn.float(), [wo])[0] + x.double(), attn
    g = _gen(seed)
    wq, wk = _norm_weights(g, d) if MODELS[model][6] else (None, None)
    if kind in ("host", "token"):
        token = case if kind == "token" else dict(case, layers=1, window=0, pattern=0)
        pos = token["position"]
        cached = [(_randn(g, pos - f, hkv * d), _randn(g, pos - f, hkv * d)) for _, _, f in _token_layers(token)]
        q, k, v = (_randn(g, token["layers"], h * d) for h in (hq, hkv, hkv))
        out = [_attend(model, q[i:i + 1], torch.cat([cached[i][0], k[i:i + 1]]),
                       torch.cat([cached[i][1], v[i:i + 1]]), pos, f, w, wq, wk)
               for i, w, f in _token_layers(token)]
        out = torch.cat(out)
        return out[0].cpu().numpy() if kind == "host" else out
    if kind == "sessions":
        lengths = _session_lengths(case, seed)
        cached = []
        for n in lengths:
            cached.append((_randn(g, int(n), hkv * d), _randn(g, int(n), hkv * d)))
        q, k, v = (_randn(g, len(lengths), h * d) for h in (hq, hkv, hkv))
        return torch.cat([_attend(model, q[s:s + 1], torch.cat([cached[s][0], k[s:s + 1]]),
                                  torch.cat([cached[s][1], v[s:s + 1]]), int(n), 0, 0, wq, wk)
                          for s, n in enumerate(lengths)])
    start, n = case["start"], case["rows"]
    ks, vs = [], []
    if start:
        ks.append(_randn(g, start, hkv * d))
        vs.append(_randn(g, start, hkv * d))
    q, k, v = (_randn(g, n, h * d) for h in (hq, hkv, hkv))
    return _attend(model, q, torch.cat(ks + [k]), torch.cat(vs + [v]), start, 0, case["window"], wq, wk)
