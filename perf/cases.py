"""Performance cases of the token loop: the calls a program makes through the public entry points.

Kinds of case:

* ``matmul``  — one projection (``engine.matmul``): f32 activations times block-quantised weights.
  M = 1 is a decode step's matvec, M > 1 a prompt's GEMM. N and K are the projection widths of the
  configurations (Mistral-7B 4096 / 1024 / 14336, Gemma-4-E2B 1536 / 6144, the tiny model's
  512 / 1408) and odd N between them.
* ``attn_decode``  — one new token's attention over a cache (``engine.attention_decode``, or
  ``attention_decode_noalloc``, the entry of serving loops and captured graphs).
* ``attn_prefill`` — a prompt's causal attention (``engine.attention_prefill``).
* ``request`` — a whole request on a session: prefill of a prompt, its logits, then ``steps`` decoded
  tokens with the logits of each (what a sampling loop reads). The decoded tokens are given, as a
  verified draft's or a replayed chat's are, so that two correct implementations cannot part ways at
  a near-tie. Models are the full widths of the configurations with fewer layers (and for Gemma-4 a
  smaller vocabulary), so that the layers keep their share of the time.
"""
from __future__ import annotations

import math
import os
import shutil
import struct
import tempfile

import numpy as np
import torch

from inference_engine_rust_amd import engine, synth

DTYPES = {"q4k": engine.Q4K, "q6k": engine.Q6K, "q8_0": engine.Q8_0, "f32": engine.F32}
BLOCK = {"q4k": (256, 144), "q6k": (256, 210), "q8_0": (32, 34)}

MODELS = {
    # Mistral-7B widths (bench's default configuration), 4 of 32 layers
    "mistral": dict(preset="c2", n_layers=4),
    # Gemma-4-E2B widths (sliding and global layers, per-layer embeddings, borrowed KV), 10 of 35 layers
    "gemma": dict(preset="c3", n_layers=10, shared_kv_layers=5, vocab=65536),
    # the tiny model: latency and launches only
    "tiny": dict(preset="c0"),
}


def listed() -> list[dict]:
    return [
        # the smallest call of a decode step: the K or V projection of one token
        dict(name="matvec_kv", kind="matmul", m=1, n=1024, k=4096, dtype="q4k"),
        # a decode step's widest reduction: the down projection, six-bit weights
        dict(name="matvec_down_q6k", kind="matmul", m=1, n=4096, k=14336, dtype="q6k"),
        # gate projection of a short chat turn (odd row count)
        dict(name="matmul_short_prompt", kind="matmul", m=23, n=14336, k=4096, dtype="q4k"),
        # FFN projection of the Gemma-4 prompt the benchmark uses
        dict(name="matmul_gemma_q8", kind="matmul", m=256, n=6144, k=1536, dtype="q8_0"),
        # down projection of the benchmark's 512-token prompt
        dict(name="matmul_down_q6k", kind="matmul", m=512, n=4096, k=14336, dtype="q6k"),
        # one token's attention in a chat of a few hundred tokens, the plain entry point
        dict(name="attn_decode_short", kind="attn_decode", heads=32, kv=8, hd=128, ctx=1024, total=531, window=0,
             cache="f32", noalloc=False),
        # one token's attention over a long context, from a serving loop
        dict(name="attn_decode_long", kind="attn_decode", heads=32, kv=8, hd=128, ctx=8704, total=8223, window=0,
             cache="f32", noalloc=True),
        # causal attention of a 2-K prompt, ragged length
        dict(name="attn_prefill_gqa", kind="attn_prefill", seq=2045, heads=32, kv=8, hd=128, window=0),
        # a Gemma-4 sliding-window layer over a prompt longer than its window
        dict(name="attn_prefill_window", kind="attn_prefill", seq=800, heads=8, kv=1, hd=256, window=512),
        # the benchmark's prompt through every layer: time to first token
        dict(name="prefill_mistral", kind="request", model="mistral", prompt=512, steps=0),
        # a chat turn: short odd prompt, then decode
        dict(name="chat_mistral", kind="request", model="mistral", prompt=19, steps=16),
        # the same on Gemma-4
        dict(name="chat_gemma", kind="request", model="gemma", prompt=67, steps=16),
    ]


def _log_uniform(rng, lo: int, hi: int) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng) -> dict:
    kind = rng.choice(["matvec", "matmul", "matmul", "attn_decode", "attn_prefill", "request", "request"])
    if kind in ("matvec", "matmul"):
        dtype = rng.choice(["q4k", "q6k", "q8_0"])
        widths = [512, 1408, 1536, 2048, 4096, 6144, 14336]
        k = rng.choice(widths)
        # whole weight tensors are whole blocks: N even where a row ends inside a superblock
        n = _log_uniform(rng, 256, 14336)
        if k % BLOCK[dtype][0]:
            n += n % 2
        m = 1 if kind == "matvec" else _log_uniform(rng, 2, 512)
        return dict(kind="matmul", m=m, n=n, k=k, dtype=dtype)
    heads, kv, hd, window = rng.choice([(32, 8, 128, 0), (8, 2, 64, 0), (8, 1, 256, 512), (8, 1, 512, 0)])
    if kind == "attn_decode":
        total = _log_uniform(rng, 4, 8704)
        ctx = min(8704, total + _log_uniform(rng, 1, 1024))
        return dict(kind=kind, heads=heads, kv=kv, hd=hd, ctx=ctx, total=total, window=window,
                    cache=rng.choice(["f32", "f32", "f16"]), noalloc=rng.choice([False, True]))
    if kind == "attn_prefill":
        return dict(kind=kind, seq=_log_uniform(rng, 4, 2045), heads=heads, kv=kv, hd=hd, window=window)
    model = rng.choice(["mistral", "mistral", "gemma", "tiny"])
    if model == "tiny":
        prompt = _log_uniform(rng, 2, 48)
        return dict(kind=kind, model=model, prompt=prompt, steps=rng.randint(0, 16))
    prompt = _log_uniform(rng, 2, 512 if model == "mistral" else 400)
    return dict(kind=kind, model=model, prompt=prompt, steps=0 if prompt > 128 else rng.randint(0, 16))


# ---- weights in GGUF blocks, made and read back with torch ----------------------------------------


def _bytes_of(x: torch.Tensor) -> torch.Tensor:
    return x.to(torch.float16).contiguous().view(torch.uint8).reshape(x.shape[0], -1)


def _quant_q8_0(w: torch.Tensor) -> torch.Tensor:
    b = w.reshape(-1, 32)
    d = (b.abs().amax(1, keepdim=True) / 127).half().float()
    q = torch.round(b / d.clamp_min(1e-12)).clamp(-127, 127).to(torch.int8)
    return torch.cat([_bytes_of(d), q.view(torch.uint8)], 1)


def _quant_q4k(w: torch.Tensor) -> torch.Tensor:
    b = w.reshape(-1, 8, 32)
    lo = (-b.amin(2)).clamp_min(0)
    scale = (b.amax(2) + lo) / 15
    d = (scale.amax(1, keepdim=True) / 63).half().float()
    dmin = (lo.amax(1, keepdim=True) / 63).half().float()
    sc = torch.round(scale / d.clamp_min(1e-12)).clamp(0, 63)
    mn = torch.round(lo / dmin.clamp_min(1e-12)).clamp(0, 63)
    q = torch.round((b + (dmin * mn)[..., None]) / (d * sc)[..., None].clamp_min(1e-12)).clamp(0, 15).to(torch.uint8)
    sc, mn = sc.to(torch.uint8), mn.to(torch.uint8)
    packed = torch.cat([sc[:, :4] | ((sc[:, 4:] >> 4) << 6), mn[:, :4] | ((mn[:, 4:] >> 4) << 6),
                        (sc[:, 4:] & 15) | ((mn[:, 4:] & 15) << 4)], 1)
    qs = (q[:, 0::2] | (q[:, 1::2] << 4)).reshape(-1, 128)
    return torch.cat([_bytes_of(d), _bytes_of(dmin), packed, qs], 1)


def _quant_q6k(w: torch.Tensor) -> torch.Tensor:
    b = w.reshape(-1, 16, 16)
    scale = b.abs().amax(2) / 31
    d = (scale.amax(1, keepdim=True) / 127).half().float()
    sc = torch.round(scale / d.clamp_min(1e-12)).clamp(1, 127)
    q = (torch.round(b / (d * sc)[..., None].clamp_min(1e-12)).clamp(-32, 31) + 32).to(torch.uint8).reshape(-1, 2, 4, 32)
    ql = torch.cat([(q[:, :, 0] & 15) | ((q[:, :, 2] & 15) << 4), (q[:, :, 1] & 15) | ((q[:, :, 3] & 15) << 4)], 2)
    qh = (q[:, :, 0] >> 4) | ((q[:, :, 1] >> 4) << 2) | ((q[:, :, 2] >> 4) << 4) | ((q[:, :, 3] >> 4) << 6)
    n = q.shape[0]
    return torch.cat([ql.reshape(n, 128), qh.reshape(n, 64), sc.to(torch.int8).view(torch.uint8), _bytes_of(d)], 1)


def _blocks(dtype: str, w: torch.Tensor) -> torch.Tensor:
    """Native GGUF bytes of a flat f32 weight (element (k, n) at k + n * K)."""
    if dtype == "f32":
        return w.contiguous().view(torch.uint8)
    return {"q4k": _quant_q4k, "q6k": _quant_q6k, "q8_0": _quant_q8_0}[dtype](w).contiguous().reshape(-1)


def _f16_at(b: torch.Tensor, at: int) -> torch.Tensor:
    return b[:, at:at + 2].contiguous().view(torch.float16).double()


def _values(dtype: str, raw: torch.Tensor) -> torch.Tensor:
    """The f64 weights the bytes stand for, flat."""
    if dtype == "f32":
        return raw.contiguous().view(torch.float32).double()
    if dtype == "bf16":
        return raw.contiguous().view(torch.bfloat16).double()
    b = raw.reshape(-1, BLOCK[dtype][1])
    n = b.shape[0]
    if dtype == "q8_0":
        return (_f16_at(b, 0) * b[:, 2:].contiguous().view(torch.int8).double()).reshape(-1)
    if dtype == "q4k":
        s = b[:, 4:16]
        sc = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | ((s[:, :4] >> 6) << 4)], 1).double()
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).double()
        qs = b[:, 16:].reshape(n, 4, 32)
        q = torch.stack([qs & 15, qs >> 4], 2).reshape(n, 8, 32).double()
        return ((_f16_at(b, 0) * sc)[..., None] * q - (_f16_at(b, 2) * mn)[..., None]).reshape(-1)
    ql, qh = b[:, :128].reshape(n, 2, 2, 32), b[:, 128:192].reshape(n, 2, 32)
    q = torch.stack([(ql[:, :, 0] & 15) | ((qh & 3) << 4), (ql[:, :, 1] & 15) | (((qh >> 2) & 3) << 4),
                     (ql[:, :, 0] >> 4) | (((qh >> 4) & 3) << 4), (ql[:, :, 1] >> 4) | ((qh >> 6) << 4)], 2)
    q = q.reshape(n, 16, 16).double() - 32
    sc = b[:, 192:208].contiguous().view(torch.int8).double()
    return ((_f16_at(b, 208) * sc)[..., None] * q).reshape(-1)


# ---- models --------------------------------------------------------------------------------------

_loaded: dict = {}


def _spec(model: str):
    over = dict(MODELS[model])
    return synth.preset(over.pop("preset"), **over)


class _File:
    """The model's GGUF, written to memory-backed storage while it is read."""

    def __init__(self, model: str):
        self.model = model

    def __enter__(self) -> str:
        self.dir = tempfile.mkdtemp(prefix="iek_cases_", dir="/dev/shm" if os.path.isdir("/dev/shm") else None)
        return synth.write_model(os.path.join(self.dir, "m.gguf"), _spec(self.model), seed=0)

    def __exit__(self, *exc):
        shutil.rmtree(self.dir, ignore_errors=True)


def _model(name: str) -> engine.LoadedModel:
    if name not in _loaded:
        with _File(name) as path:
            _loaded[name] = engine.LoadedModel.load(path, device=0)
    return _loaded[name]


# ---- the calls -----------------------------------------------------------------------------------


def _gen(seed: int) -> torch.Generator:
    return torch.Generator(device="cuda").manual_seed(seed)


def prepare(case: dict, seed: int) -> dict:
    c = case
    if c["kind"] == "request":
        vocab = _spec(c["model"]).vocab
        ids = np.random.default_rng(seed).integers(3, vocab, c["prompt"] + c["steps"]).astype(np.uint32)
        return dict(c, session=engine.InferenceSession(_model(c["model"])), ids=ids[:c["prompt"]],
                    forced=[int(t) for t in ids[c["prompt"]:]])
    g = _gen(seed)
    rand = lambda *shape: torch.randn(*shape, generator=g, device="cuda")  # noqa: E731
    if c["kind"] == "matmul":
        w = _blocks(c["dtype"], rand(c["n"] * c["k"]).mul_(0.02))
        return dict(c, w=w, x=rand(c["m"], c["k"]), out=torch.empty(c["m"], c["n"], device="cuda"))
    if c["kind"] == "attn_decode":
        dt = torch.float16 if c["cache"] == "f16" else torch.float32
        return dict(c, q=rand(c["heads"], c["hd"]), kc=rand(c["kv"], c["ctx"], c["hd"]).to(dt),
                    vc=rand(c["kv"], c["ctx"], c["hd"]).to(dt), scale=_scale(c),
                    out=torch.empty(c["heads"], c["hd"], device="cuda"))
    return dict(c, q=rand(c["seq"], c["heads"], c["hd"]), k=rand(c["seq"], c["kv"], c["hd"]),
                v=rand(c["seq"], c["kv"], c["hd"]), scale=_scale(c),
                out=torch.empty(c["seq"], c["heads"], c["hd"], device="cuda"))


def _scale(c: dict) -> float:
    return 1.0 / math.sqrt(c["hd"])


def run(state: dict):
    s = state
    if s["kind"] == "request":
        session = s["session"]
        session.reset()
        session.prefill(s["ids"])
        logits = [session.logits_last_token()]
        for t in s["forced"]:
            session.decode_token(t)
            logits.append(session.logits_last_token())
        return logits
    stream = torch.cuda.current_stream().cuda_stream
    if s["kind"] == "matmul":
        engine.matmul(s["x"].data_ptr(), s["m"], s["k"], DTYPES[s["dtype"]], s["w"].data_ptr(), s["w"].numel(), s["n"],
                      s["out"].data_ptr(), stream)
    elif s["kind"] == "attn_decode":
        entry = engine.attention_decode_noalloc if s["noalloc"] else engine.attention_decode
        entry(s["q"].data_ptr(), s["kc"].data_ptr(), s["vc"].data_ptr(),
              engine.F16 if s["cache"] == "f16" else engine.F32, s["heads"], s["kv"], s["hd"], s["ctx"], s["total"],
              s["window"], s["scale"], s["out"].data_ptr(), stream)
    else:
        engine.attention_prefill(s["q"].data_ptr(), s["k"].data_ptr(), s["v"].data_ptr(), s["seq"], s["heads"], s["kv"],
                                 s["hd"], s["window"], s["scale"], s["out"].data_ptr(), stream)
    return s["out"]


# ---- what a pass cannot do without ---------------------------------------------------------------


def _weight_bytes(dtype: str, elems: int) -> float:
    if dtype in ("f32", "bf16"):  # bf16 tensors are held as f32
        return 4.0 * elems
    be, bb = BLOCK[dtype]
    return elems / be * bb


def _pairs(rows: int, window: int, past: int = 0) -> int:
    """(query, key) pairs of `rows` causal rows after `past` earlier keys."""
    return sum(min(past + p + 1, window) if window > 0 else past + p + 1 for p in range(rows))


_NAMES = {synth.GGML_F32: "f32", synth.GGML_Q4_K: "q4k", synth.GGML_Q6_K: "q6k", synth.GGML_Q8_0: "q8_0",
          synth.GGML_BF16: "bf16"}


def _layers(model: str):
    """Per layer: (matmul weights as (dtype, K, N)), head dim, window, whether it writes its own KV."""
    s = _spec(model)
    out = []
    for li in range(s.n_layers):
        if isinstance(s, synth.GemmaSpec):
            hd, own = s.head_dim(li), li < s.n_layers - s.shared_kv_layers
            t = _NAMES[s.t_weights]
            qd, kvd = s.n_heads * hd, s.n_kv_heads * hd
            ws = [(t, s.hidden, qd), (t, qd, s.hidden), (t, s.hidden, s.ffn), (t, s.hidden, s.ffn), (t, s.ffn, s.hidden),
                  (t, s.hidden, s.ple_dim), (t, s.ple_dim, s.hidden)] + [(t, s.hidden, kvd)] * (2 if own else 0)
            out.append((ws, hd, s.sliding_window if s.is_swa(li) else 0, own))
        else:
            a, g, d = _NAMES[s.t_attn], _NAMES[s.t_ffn_gate_up], _NAMES[s.t_ffn_down]
            kvd = s.n_kv_heads * s.head_dim
            ws = [(a, s.hidden, s.hidden), (a, s.hidden, kvd), (a, s.hidden, kvd), (a, s.hidden, s.hidden),
                  (g, s.hidden, s.ffn), (g, s.hidden, s.ffn), (d, s.ffn, s.hidden)]
            out.append((ws, s.head_dim, 0, True))
    return s, out


def work(case: dict) -> dict:
    c = case
    if c["kind"] == "matmul":
        m, n, k = c["m"], c["n"], c["k"]
        return dict(bytes=_weight_bytes(c["dtype"], n * k) + 4.0 * m * (n + k), flops=2.0 * m * n * k)
    if c["kind"] == "attn_decode":
        keys = min(c["total"], c["window"]) if c["window"] else c["total"]
        esz = 2 if c["cache"] == "f16" else 4
        return dict(bytes=2.0 * c["kv"] * keys * c["hd"] * esz + 8.0 * c["heads"] * c["hd"],
                    flops=4.0 * c["heads"] * keys * c["hd"])
    if c["kind"] == "attn_prefill":
        return dict(bytes=4.0 * c["seq"] * c["hd"] * 2 * (c["heads"] + c["kv"]),
                    flops=4.0 * c["heads"] * c["hd"] * _pairs(c["seq"], c["window"]))
    s, layers = _layers(c["model"])
    gemma = isinstance(s, synth.GemmaSpec)
    n, steps = c["prompt"], c["steps"]
    by = fl = 0.0
    for ws, hd, window, own in layers:
        for t, k, w in ws:
            by += (1 + steps) * _weight_bytes(t, k * w)
            fl += 2.0 * k * w * (n + steps)
        row = 2.0 * s.n_kv_heads * hd * 4
        by += row * (n + steps) * (1 if own else 0) + row * _pairs(steps, window, n)
        fl += 4.0 * s.n_heads * hd * (_pairs(n, window) + _pairs(steps, window, n))
    if gemma:
        packn = s.n_layers * s.ple_dim
        by += (1 + steps) * 4.0 * s.hidden * packn
        fl += 2.0 * s.hidden * packn * (n + steps)
    head = _NAMES[s.t_embd if gemma else s.t_output]
    by += (1 + steps) * (_weight_bytes(head, s.hidden * s.vocab) + 4.0 * s.vocab)
    fl += (1 + steps) * 2.0 * s.hidden * s.vocab
    return dict(bytes=by, flops=fl)


def tolerance(case: dict):
    """Relative 2-norm bounds, about four times the largest distance from 64 bits measured: single
    calls 1e-7 to 4e-7 (f32 sums; operands as fp16 pairs of 22 bits), the logits of 4 Mistral layers
    4e-6, of 10 Gemma-4 layers 2e-4 (random weights amplify rounding there)."""
    if case["kind"] != "request":
        return {"rel": 2e-6}
    return {"rel": 1e-3 if case["model"] == "gemma" else 1.5e-5}


# ---- the same in 64 bits -------------------------------------------------------------------------


def _attention(q, k, v, heads, kv, hd, window, scale):
    """q [m, heads, hd], k and v [m, kv, hd]: causal attention with an optional sliding window."""
    m = q.shape[0]
    p = torch.arange(m, device=q.device)
    mask = p[None, :] <= p[:, None]
    if window > 0:
        mask &= p[None, :] >= p[:, None] - (window - 1)
    out = torch.empty(m, heads, hd, dtype=torch.float64, device=q.device)
    for h in range(heads):
        kh = h // (heads // kv)
        sc = (q[:, h] @ k[:, kh].T * scale).masked_fill(~mask, -math.inf)
        out[:, h] = torch.softmax(sc, 1) @ v[:, kh]
    return out


def exact(case: dict, seed: int):
    c = case
    if c["kind"] == "request":
        return _exact_request(c, seed)
    s = prepare(c, seed)
    if c["kind"] == "matmul":
        out = torch.empty(c["m"], c["n"], dtype=torch.float64, device="cuda")
        w = _values(c["dtype"], s["w"]).reshape(c["n"], c["k"])
        torch.matmul(s["x"].double(), w.T, out=out)
        return out
    if c["kind"] == "attn_decode":
        lo = max(0, c["total"] - c["window"]) if c["window"] else 0
        k, v = s["kc"][:, lo:c["total"]].double(), s["vc"][:, lo:c["total"]].double()
        q = s["q"].double().reshape(c["kv"], c["heads"] // c["kv"], c["hd"])
        out = [torch.softmax(q[h] @ k[h].T * c_scale, 1) @ v[h] for c_scale in [s["scale"]] for h in range(c["kv"])]
        return torch.cat(out)
    return _attention(s["q"].double(), s["k"].double(), s["v"].double(), c["heads"], c["kv"], c["hd"], c["window"],
                      s["scale"])


class _Tensors:
    """Tensors of a GGUF file, as f64 on the GPU when asked for."""

    def __init__(self, path: str):
        self.data = np.memmap(path, np.uint8, "r")
        head = self.data[:1 << 24].tobytes()
        _, _, n_t, n_kv = struct.unpack_from("<IIQQ", head, 0)
        at = 24
        for _ in range(n_kv):
            at = self._skip_string(head, at)
            (t,) = struct.unpack_from("<I", head, at)
            at = self._skip_value(head, at + 4, t)
        self.info = {}
        for _ in range(n_t):
            end = self._skip_string(head, at)
            name = head[at + 8:end].decode()
            (nd,) = struct.unpack_from("<I", head, end)
            dims = struct.unpack_from(f"<{nd}Q", head, end + 4)
            t, off = struct.unpack_from("<IQ", head, end + 4 + 8 * nd)
            at = end + 4 + 8 * nd + 12
            self.info[name] = (_NAMES[t], dims, off)
        self.base = -(-at // 32) * 32

    @staticmethod
    def _skip_string(b, at):
        return at + 8 + struct.unpack_from("<Q", b, at)[0]

    @classmethod
    def _skip_value(cls, b, at, t):
        if t == 8:
            return cls._skip_string(b, at)
        if t == 9:
            et, n = struct.unpack_from("<IQ", b, at)
            at += 12
            for _ in range(n):
                at = cls._skip_value(b, at, et)
            return at
        return at + {0: 1, 1: 1, 2: 2, 3: 2, 4: 4, 5: 4, 6: 4, 7: 1, 10: 8, 11: 8, 12: 8}[t]

    def rows(self, name: str, ids=None) -> torch.Tensor:
        t, dims, off = self.info[name]
        k = dims[0]
        n = dims[1] if len(dims) > 1 else 1
        per = int(_weight_bytes(t, k)) if t != "bf16" else 2 * k
        raw = self.data[self.base + off:self.base + off + per * n]
        if ids is not None:
            raw = raw.reshape(n, per)[np.asarray(ids, np.int64)].reshape(-1)
            n = len(ids)
        return _values(t, torch.from_numpy(np.array(raw)).cuda()).reshape(n, k)

    def vec(self, name: str) -> torch.Tensor:
        return self.rows(name)[0]


def _rms(x, eps, w=None):
    y = x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)
    return y if w is None else y * w


def _rope(x, theta, rot):
    """x [m, heads, hd]; adjacent pairs; the angles are the f32 running products the models use."""
    m = x.shape[0]
    step = np.float32(np.float32(theta) ** np.float32(-2.0 / rot))
    ang = np.empty((m, rot // 2), np.float32)
    t = np.arange(m, dtype=np.float32)
    for i in range(rot // 2):
        ang[:, i] = t
        t = t * step
    a = torch.from_numpy(ang).cuda().double()[:, None, :]
    even, odd = x[..., 0:rot:2].clone(), x[..., 1:rot:2].clone()
    y = x.clone()
    y[..., 0:rot:2] = even * torch.cos(a) - odd * torch.sin(a)
    y[..., 1:rot:2] = even * torch.sin(a) + odd * torch.cos(a)
    return y


def _exact_request(c: dict, seed: int):
    spec = _spec(c["model"])
    ids = np.random.default_rng(seed).integers(3, spec.vocab, c["prompt"] + c["steps"])
    with _File(c["model"]) as path:
        T = _Tensors(path)
        x = _exact_gemma(spec, T, ids) if isinstance(spec, synth.GemmaSpec) else _exact_llama(spec, T, ids)
        x = _rms(x[c["prompt"] - 1:], spec.rms_eps, T.vec("output_norm.weight"))
        head = "token_embd.weight" if "output.weight" not in T.info else "output.weight"
        z = torch.cat([x @ T.rows(head, np.arange(a, min(a + 8192, spec.vocab))).T
                       for a in range(0, spec.vocab, 8192)], 1)
        if getattr(spec, "softcap", 0):
            z = spec.softcap * torch.tanh(z / spec.softcap)
        return [r for r in z]


def _exact_llama(s, T, ids):
    m = len(ids)
    x = T.rows("token_embd.weight", ids)
    for li in range(s.n_layers):
        w = lambda n: T.rows(f"blk.{li}.{n}.weight")  # noqa: E731
        a = _rms(x, s.rms_eps, w("attn_norm")[0])
        q = _rope((a @ w("attn_q").T).reshape(m, s.n_heads, s.head_dim), s.rope_theta, s.head_dim)
        k = _rope((a @ w("attn_k").T).reshape(m, s.n_kv_heads, s.head_dim), s.rope_theta, s.head_dim)
        v = (a @ w("attn_v").T).reshape(m, s.n_kv_heads, s.head_dim)
        o = _attention(q, k, v, s.n_heads, s.n_kv_heads, s.head_dim, 0, 1.0 / math.sqrt(s.head_dim))
        x = x + o.reshape(m, -1) @ w("attn_output").T
        f = _rms(x, s.rms_eps, w("ffn_norm")[0])
        x = x + (torch.nn.functional.silu(f @ w("ffn_gate").T) * (f @ w("ffn_up").T)) @ w("ffn_down").T
    return x


def _exact_gemma(s, T, ids):
    m, eps, pd = len(ids), s.rms_eps, s.ple_dim
    gelu = lambda t: torch.nn.functional.gelu(t, approximate="tanh")  # noqa: E731
    x = T.rows("token_embd.weight", ids) * math.sqrt(s.hidden)
    proj = (x @ T.rows("per_layer_model_proj.weight").T / math.sqrt(s.hidden)).reshape(m, s.n_layers, pd)
    tok = T.rows("per_layer_token_embd.weight", ids).reshape(m, s.n_layers, pd) * math.sqrt(pd)
    packed = (_rms(proj, eps, T.vec("per_layer_proj_norm.weight")) + tok) / math.sqrt(2.0)
    kvs = {}
    own = s.n_layers - s.shared_kv_layers
    for li in range(s.n_layers):
        w = lambda n: T.rows(f"blk.{li}.{n}.weight")  # noqa: E731
        swa, hd = s.is_swa(li), s.head_dim(li)
        theta, rot = (s.theta_swa, s.rot_swa) if swa else (s.theta_global, s.rot_global)
        a = _rms(x, eps, w("attn_norm")[0])
        q = _rms((a @ w("attn_q").T).reshape(m, s.n_heads, hd), eps, w("attn_q_norm")[0])
        q = _rope(q, theta, rot)
        if li < own:
            k = _rms((a @ w("attn_k").T).reshape(m, s.n_kv_heads, hd), eps, w("attn_k_norm")[0])
            kvs[li] = (_rope(k, theta, rot), _rms((a @ w("attn_v").T).reshape(m, s.n_kv_heads, hd), eps))
            k, v = kvs[li]
        else:  # the last layer of its kind that keeps a cache
            k, v = kvs[max(j for j in range(own) if s.is_swa(j) == swa)]
        o = _attention(q, k, v, s.n_heads, s.n_kv_heads, hd, s.sliding_window if swa else 0, 1.0)
        x = x + _rms(o.reshape(m, -1) @ w("attn_output").T, eps, w("post_attention_norm")[0])
        f = _rms(x, eps, w("ffn_norm")[0])
        f = (gelu(f @ w("ffn_gate").T) * (f @ w("ffn_up").T)) @ w("ffn_down").T
        x = x + _rms(f, eps, w("post_ffw_norm")[0])
        p = (gelu(x @ w("inp_gate").T) * packed[:, li]) @ w("proj").T
        x = (x + _rms(p, eps, w("post_norm")[0])) * w("layer_output_scale").reshape(-1)[0]
    return x
