"""The calls whose time matters to a user of this framework, as cases that can be prepared, run and checked.

A case is one call (or one short conversation) through the public Python API: a quantized mat-mul of some
activation rows, attention over an f16 KV cache, the encoding of a weight, or a decoder answering a
prompt. The listed cases and the drawn ones cover the same ranges: one row (decode), a few (batched
decode), tens (a short prompt or speculative rows), hundreds and thousands (a prompt chunk); weights in
each storage type; the 8B-shaped decoder's projections and sizes that are no multiple of a tile.

Weights are given as the block bytes a GGUF file holds (encoded here by plain rounding, not by the
framework's encoders) and uploaded once, as a loader does.
"""

from __future__ import annotations

import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ggml-compiler_amd"))

from ggml_compiler_amd import ops  # noqa: E402
from ggml_compiler_amd.llm import LlamaConfig, Model  # noqa: E402

EPS = 1e-5
BLOCK_BYTES = {"q4_0": (32, 18), "q8_0": (32, 34), "q4_K": (256, 144), "q5_K": (256, 176), "q6_K": (256, 210)}
KQ = ("q4_K", "q5_K", "q6_K")


# ------------------------------------------------------------------------------------------ cases


def listed() -> list[dict]:
    return [
        # One decode row through the attention output projection: the smallest mat-mul of a decoder layer.
        {"name": "row_q4_0", "kind": "mul_mat", "type": "q4_0", "M": 1, "N": 4096, "K": 4096},
        # The decode step's largest layer weight, gate and up stacked, with the rms_norm in front of it.
        {"name": "norm_gate_up_q4_0", "kind": "norm_mul_mat", "type": "q4_0", "M": 1, "N": 28672, "K": 4096},
        # The lm head of a Q4_K_M file (Q6_K), one row: the longest single read of a decode step.
        {"name": "lm_head_q6_K", "kind": "mul_mat", "type": "q6_K", "M": 1, "N": 128256, "K": 4096},
        # Five sequences decoded together through the stacked q / k / v projection.
        {"name": "batch5_q4_K", "kind": "mul_mat", "type": "q4_K", "M": 5, "N": 6144, "K": 4096},
        # A short prompt (33 tokens) through the down projection.
        {"name": "short_prompt_q4_0", "kind": "mul_mat", "type": "q4_0", "M": 33, "N": 4096, "K": 14336},
        # A 512-token prompt chunk, Q8_0, one of the feed-forward projections.
        {"name": "prompt_q8_0", "kind": "mul_mat", "type": "q8_0", "M": 512, "N": 14336, "K": 4096},
        # A long prompt in one call (an odd 1999 rows), Q4_K.
        {"name": "long_prompt_q4_K", "kind": "mul_mat", "type": "q4_K", "M": 1999, "N": 14336, "K": 4096},
        # A decode step's attention at a 4096-token context.
        {"name": "attn_decode_4096", "kind": "attention", "H": 32, "Hkv": 8, "D": 128, "Sq": 1, "n_kv": 4096,
         "ctx": 4096, "past": 4095, "mask": False},
        # The attention of a 512-token chunk late in a long prompt, causal.
        {"name": "attn_chunk_4096", "kind": "attention", "H": 32, "Hkv": 8, "D": 128, "Sq": 512, "n_kv": 4096,
         "ctx": 8192, "past": 3584, "mask": True},
        # A short prompt's attention from an empty context in a small model: 7 query heads per KV head of 64,
        # rows padded as the compiled programs pad the KV length (to a multiple of 256).
        {"name": "attn_short_prompt", "kind": "attention", "H": 14, "Hkv": 2, "D": 64, "Sq": 129, "n_kv": 256,
         "ctx": 1024, "past": 0, "mask": True},
        # Storing an f32 weight as Q4_K (ggml_compiler_quantize): the down projection.
        {"name": "encode_q4_K", "kind": "quantize", "type": "q4_K", "N": 4096, "K": 14336},
        # A conversation turn on an 8B-shaped decoder cut to two layers: a 500-token prompt, then 16 tokens one
        # by one with their logits, as a host-side sampling loop reads them.
        {"name": "turn_2_layers", "kind": "model", "layers": 2, "prompt": 500, "steps": 16, "wtype": "q4_0"},
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng) -> dict:
    """One more case of the listed ranges, its sizes spread over their logarithm, odd ones among them."""
    kind = rng.choice(["row", "norm", "batch", "short", "prompt", "prompt", "attn1", "attn", "attn", "quantize", "model"])
    if kind in ("row", "norm", "batch", "short", "prompt"):
        t = rng.choice(["q4_0", "q8_0"]) if kind == "norm" else rng.choice(list(BLOCK_BYTES))
        step = BLOCK_BYTES[t][0] if rng.random() < 0.5 else 1024
        K = max(1024, _log_int(rng, 1024, 14336) // step * step)
        N = _log_int(rng, 1024, 32768)
        if rng.random() < 0.5:
            N = max(1, N // 128) * 128
        M = {"row": 1, "norm": 1, "batch": rng.randint(2, 8), "short": _log_int(rng, 9, 128),
             "prompt": _log_int(rng, 129, 2048)}[kind]
        while M * N * K > 1999 * 14336 * 4096:
            N = (N + 1) // 2
        return {"kind": "norm_mul_mat" if kind == "norm" else "mul_mat", "type": t, "M": M, "N": N, "K": K}
    if kind in ("attn1", "attn"):
        D = rng.choice([64, 128, 128])
        G = rng.choice([1, 2, 4, 4, 7, 8]) if kind == "attn" else rng.choice([1, 2, 4, 8])
        Hkv = rng.choice([2, 4, 8])
        Sq = 1 if kind == "attn1" else _log_int(rng, 2, 1024)
        limit = 32768 if kind == "attn1" else max(64, 512 * 4096 * 32 * 128 // (Sq * G * Hkv * D))
        past = _log_int(rng, 1, max(2, min(limit, 32768) - Sq)) - 1 if Sq < limit else 0
        used = past + Sq
        pad = kind == "attn" and rng.random() < 0.5
        n_kv = (used + 255) // 256 * 256 if pad else used
        return {"kind": "attention", "H": G * Hkv, "Hkv": Hkv, "D": D, "Sq": Sq, "n_kv": n_kv,
                "ctx": n_kv + rng.choice([0, 0, 96, 1000]), "past": past, "mask": kind == "attn" or rng.random() < 0.3}
    if kind == "quantize":
        t = rng.choice(list(BLOCK_BYTES))
        K = max(1, _log_int(rng, 1024, 14336) // 256) * 256
        return {"kind": "quantize", "type": t, "N": _log_int(rng, 64, 4096), "K": K}
    return {"kind": "model", "layers": rng.choice([1, 2]), "prompt": _log_int(rng, 2, 500), "steps": rng.randint(1, 16),
            "wtype": "q4_0"}


# ------------------------------------------------------------------------- inputs (plain torch)


def _gen(seed: int, what: int) -> torch.Generator:
    g = torch.Generator(device="cuda")
    g.manual_seed((seed * 1000003 + what) % (1 << 62))
    return g


def _normal(shape, seed: int, what: int, std: float = 1.0) -> torch.Tensor:
    return torch.randn(shape, generator=_gen(seed, what), device="cuda", dtype=torch.float32) * std


def _bytes16(x: torch.Tensor) -> torch.Tensor:
    """f16 [n] as bytes [n, 2]."""
    return x.to(torch.float16).reshape(-1, 1).view(torch.uint8)


def _inv(x: torch.Tensor) -> torch.Tensor:
    return torch.where(x == 0, torch.zeros_like(x), 1.0 / x)


def _encode(w: torch.Tensor, t: str, values: bool = False):
    """f32 rows as block bytes by plain rounding: uint8 [N, row bytes], or with `values` what they decode to
    (f64 [N, K])."""
    N, K = w.shape
    if t == "q8_0":
        x = w.reshape(-1, 32)
        d = (x.abs().amax(1, keepdim=True) / 127).half().float()
        q = torch.round(x * _inv(d)).clamp(-127, 127)
        if values:
            return (q.double() * d.double()).reshape(N, K)
        return torch.cat([_bytes16(d), q.to(torch.int8).view(torch.uint8)], 1).reshape(N, -1)
    if t == "q4_0":
        x = w.reshape(-1, 32)
        d = (x.abs().amax(1, keepdim=True) / 7.5).half().float()
        q = torch.round(x * _inv(d)).clamp(-8, 7)
        if values:
            return (q.double() * d.double()).reshape(N, K)
        b = (q + 8).to(torch.uint8)
        return torch.cat([_bytes16(d), b[:, :16] | (b[:, 16:] << 4)], 1).reshape(N, -1)
    x = w.reshape(-1, 256)
    n = x.shape[0]
    if t == "q6_K":
        s = x.reshape(n, 16, 16)
        a = s.abs().amax(2) / 31
        d = (a.amax(1, keepdim=True) / 127).half().float()
        sc = torch.round(a * _inv(d)).clamp(0, 127)
        step = (sc * d).unsqueeze(2)
        q = torch.round(s * _inv(step)).clamp(-32, 31)
        if values:
            return (q.double() * sc.double().unsqueeze(2) * d.double().unsqueeze(2)).reshape(N, K)
        b = (q + 32).to(torch.uint8).reshape(n, 2, 4, 32)  # half, quarter of 32 values
        lo, hi = b & 15, b >> 4
        ql = torch.cat([lo[:, :, 0] | (lo[:, :, 2] << 4), lo[:, :, 1] | (lo[:, :, 3] << 4)], 2).reshape(n, 128)
        qh = (hi[:, :, 0] | (hi[:, :, 1] << 2) | (hi[:, :, 2] << 4) | (hi[:, :, 3] << 6)).reshape(n, 64)
        return torch.cat([ql, qh, sc.to(torch.int8).view(torch.uint8), _bytes16(d)], 1).reshape(N, -1)
    top = 15 if t == "q4_K" else 31
    s = x.reshape(n, 8, 32)
    lowest = s.amin(2).clamp(max=0)
    scale = (s.amax(2).clamp(min=0) - lowest) / top
    d = (scale.amax(1, keepdim=True) / 63).half().float()
    dm = ((-lowest).amax(1, keepdim=True) / 63).half().float()
    sc = torch.round(scale * _inv(d)).clamp(0, 63)
    mn = torch.round(-lowest * _inv(dm)).clamp(0, 63)
    q = torch.round((s + (mn * dm).unsqueeze(2)) * _inv((sc * d).unsqueeze(2))).clamp(0, top)
    if values:
        v = q.double() * (sc.double() * d.double()).unsqueeze(2) - (mn.double() * dm.double()).unsqueeze(2)
        return v.reshape(N, K)
    sb, mb, b = sc.to(torch.uint8), mn.to(torch.uint8), q.to(torch.uint8)
    packed = torch.cat([sb[:, :4] | ((sb[:, 4:] >> 4) << 6), mb[:, :4] | ((mb[:, 4:] >> 4) << 6),
                        (sb[:, 4:] & 15) | ((mb[:, 4:] & 15) << 4)], 1)
    lo = (b & 15).reshape(n, 4, 2, 32)
    parts = [_bytes16(d), _bytes16(dm), packed]
    if t == "q5_K":
        bits = torch.arange(8, device=b.device, dtype=torch.uint8).reshape(1, 8, 1)
        parts.append(((b >> 4) << bits).sum(1, dtype=torch.uint8))
    parts.append((lo[:, :, 0] | (lo[:, :, 1] << 4)).reshape(n, 128))
    return torch.cat(parts, 1).reshape(N, -1)


def _weight_f32(N: int, K: int, seed: int, what: int) -> torch.Tensor:
    return _normal((N, K), seed, what, 0.02)


def _rows(case: dict, seed: int) -> torch.Tensor:
    """Activation rows: N(0, 1) with a few channels ten times larger, as hidden states have them."""
    x = _normal((case["M"], case["K"]), seed, 2)
    x[:, 7::509] *= 10.0
    return x


def _attention_inputs(case: dict, seed: int):
    H, Hkv, D, Sq, ctx, n_kv = (case[k] for k in ("H", "Hkv", "D", "Sq", "ctx", "n_kv"))
    q = _normal((Sq, H, D), seed, 3).transpose(0, 1)  # [H, Sq, D], as a projection's rows are viewed
    k = _normal((Hkv, ctx, D), seed, 4).half()
    v = _normal((Hkv, ctx, D), seed, 5).half()
    mask = None
    if case["mask"]:
        pos = case["past"] + torch.arange(Sq, device="cuda").unsqueeze(1)
        seen = torch.arange(n_kv, device="cuda").unsqueeze(0) <= pos
        mask = torch.where(seen, 0.0, -math.inf).half()
    return q, k, v, mask


def _config(case: dict) -> LlamaConfig:
    return LlamaConfig(case["layers"], 4096, 32, 8, 128, 14336, 32000, 1024, ops.type_id(case["wtype"]), EPS, 500000.0)


def _model_shapes(c: LlamaConfig) -> list[tuple[str, int, int]]:
    out = [("token_embd", c.n_vocab, c.n_embd)]
    for i in range(c.n_layer):
        out += [(f"blk.{i}.attn_qkv", c.qkv_dim, c.n_embd), (f"blk.{i}.attn_output", c.n_embd, c.n_head * c.head_dim),
                (f"blk.{i}.ffn_gate_up", 2 * c.n_ff, c.n_embd), (f"blk.{i}.ffn_down", c.n_embd, c.n_ff)]
    return out + [("output", c.n_vocab, c.n_embd)]


def _tokens(case: dict, seed: int, vocab: int) -> tuple[list[int], list[int]]:
    ids = np.random.default_rng(seed).integers(0, vocab, case["prompt"] + case["steps"]).tolist()
    return ids[:case["prompt"]], ids[case["prompt"]:]


def prepare(case: dict, seed: int):
    kind = case["kind"]
    if kind in ("mul_mat", "norm_mul_mat"):
        w = _weight_f32(case["N"], case["K"], seed, 1)
        qw = ops.QuantWeight.from_ggml(_encode(w, case["type"]), case["type"], case["K"])
        st = {"kind": kind, "w": qw, "x": _rows(case, seed)}
        if kind == "norm_mul_mat":
            st["norm"] = 1.0 + _normal((case["K"],), seed, 6, 0.1)
        return st
    if kind == "attention":
        q, k, v, mask = _attention_inputs(case, seed)
        return {"kind": kind, "q": q, "k": k, "v": v, "mask": mask, "n_kv": case["n_kv"], "scale": case["D"] ** -0.5}
    if kind == "quantize":
        return {"kind": kind, "w": _weight_f32(case["N"], case["K"], seed, 1), "type": case["type"]}
    cfg = _config(case)
    m = Model(cfg, max_prompt=512)
    for i, (name, n, k) in enumerate(_model_shapes(cfg)):
        m.set_weight(name, _encode(_weight_f32(n, k, seed, 10 + i), case["wtype"]).cpu().numpy())
    prompt, rest = _tokens(case, seed, cfg.n_vocab)
    return {"kind": kind, "model": m, "prompt": prompt, "rest": rest}


def run(state):
    kind = state["kind"]
    if kind == "mul_mat":
        return ops.mul_mat(state["w"], state["x"])
    if kind == "norm_mul_mat":
        return ops.rms_norm_mul_mat(state["w"], state["x"], state["norm"], EPS)
    if kind == "attention":
        return ops.flash_attn_ext(state["q"], state["k"], state["v"], state["mask"], state["scale"], n_kv=state["n_kv"])
    if kind == "quantize":
        return ops.quantize(state["w"], state["type"])
    m = state["model"]
    m.reset()
    out = [m.prefill(state["prompt"])]
    for t in state["rest"]:
        out.append(m.decode(t)[0])
    return np.stack(out)


# ------------------------------------------------------------------------- work and exactness


def _wbytes(t: str, n: int) -> int:
    per, size = BLOCK_BYTES[t]
    return n // per * size


def work(case: dict) -> dict:
    kind = case["kind"]
    if kind in ("mul_mat", "norm_mul_mat"):
        M, N, K = case["M"], case["N"], case["K"]
        return {"bytes": _wbytes(case["type"], N * K) + 4 * M * (K + N) + (4 * K if kind == "norm_mul_mat" else 0),
                "flops": 2 * M * N * K}
    if kind == "attention":
        H, Hkv, D, Sq, n_kv, past = (case[k] for k in ("H", "Hkv", "D", "Sq", "n_kv", "past"))
        used = past + Sq
        pairs = Sq * past + Sq * (Sq + 1) // 2 if case["mask"] else Sq * n_kv
        keys = used if case["mask"] else n_kv
        return {"bytes": 4 * keys * Hkv * D + 8 * Sq * H * D + (2 * Sq * n_kv if case["mask"] else 0),
                "flops": 4 * pairs * H * D}
    if kind == "quantize":
        n = case["N"] * case["K"]
        return {"bytes": 4 * n + _wbytes(case["type"], n), "flops": 0}
    c = _config(case)
    P, T = case["prompt"], case["steps"]
    per_layer = c.n_embd * (c.qkv_dim + c.n_head * c.head_dim + 3 * c.n_ff)
    head = c.n_vocab * c.n_embd
    layers = per_layer * c.n_layer
    pairs = (P + T) * (P + T + 1) // 2
    row = 2 * c.n_head_kv * c.head_dim * 2 * c.n_layer  # one position's K and V
    kv = row * (P + sum(P + i + 1 for i in range(T)))
    return {"bytes": (1 + T) * (_wbytes(case["wtype"], layers + head) + 4 * c.n_vocab) + kv,
            "flops": 2 * (P + T) * layers + 2 * (1 + T) * head + 4 * pairs * c.n_head * c.head_dim * c.n_layer}


def tolerance(case: dict):
    kind = case["kind"]
    if kind == "quantize":
        return "exact"  # block bytes: the encoding is defined to the bit
    if kind == "mul_mat":
        return {"rel": 2e-6}  # f32 sums of exact block products
    if kind == "norm_mul_mat":
        return {"rel": 3e-4}  # a last-bit difference of the normalized row moves a code here and there
    if kind == "attention":
        return {"rel": 2e-6}  # f32 softmax and sums over f16 keys and values
    return {"rel": 3e-2, "max": 0.3}  # 8-bit activation codes at every projection: one row order against another, 1.6e-2


def _act_q8_0(x: torch.Tensor) -> torch.Tensor:
    """Rows as their Q8_0 blocks decode (d kept in f16, codes from the f32 scale), f64."""
    b = x.reshape(-1, 32)
    a = b.abs().amax(1, keepdim=True)
    q = torch.round(b * (127.0 * _one(a) / a).where(a != 0, torch.zeros_like(a)))
    return (q.double() * (a / (127.0 * _one(a))).half().double()).reshape(x.shape)


def _one(a: torch.Tensor) -> torch.Tensor:
    return torch.ones_like(a)


def _act_q8_K(x: torch.Tensor) -> torch.Tensor:
    """Rows as their Q8_K super-blocks decode (scale from the signed value of largest magnitude), f64."""
    b = x.reshape(-1, 256)
    top = b.gather(1, b.abs().argmax(1, keepdim=True))
    inv = (-127.0 * _one(top) / top).where(top != 0, torch.zeros_like(top))
    q = torch.round(b * inv).clamp(max=127)
    return (q.double() * (1.0 / inv).double()).where(top != 0, torch.zeros_like(q, dtype=torch.float64)).reshape(x.shape)


def _product(x: torch.Tensor, t: str, N: int, K: int, seed: int, what: int) -> torch.Tensor:
    """x [M, K] (f64) times the decoded weight's rows, in slices of rows."""
    w = _weight_f32(N, K, seed, what)
    return torch.cat([x @ _encode(w[i:i + 4096], t, values=True).T for i in range(0, N, 4096)], 1)


def _attend(q, k, v, mask, scale):
    """Softmax attention in f64, q [H, Sq, D], k / v [Hkv, n, D] -> [Sq, H, D]; rows of G heads at a time."""
    H, Sq, D = q.shape
    G = H // k.shape[0]
    out = torch.empty((Sq, H, D), dtype=torch.float64, device=q.device)
    for h in range(H):
        s = (q[h] @ k[h // G].T.contiguous()) * scale
        if mask is not None:
            s = s + mask
        out[:, h] = torch.softmax(s, 1) @ v[h // G]
    return out


def exact(case: dict, seed: int):
    kind = case["kind"]
    if kind == "quantize":
        return None
    if kind in ("mul_mat", "norm_mul_mat"):
        x = _rows(case, seed)
        if kind == "norm_mul_mat":
            scale = 1.0 / torch.sqrt((x * x).double().mean(1, keepdim=True).float() + EPS)
            x = x * scale * (1.0 + _normal((case["K"],), seed, 6, 0.1))
        x = _act_q8_K(x) if case["type"] in KQ else _act_q8_0(x)
        return _product(x, case["type"], case["N"], case["K"], seed, 1)
    if kind == "attention":
        q, k, v, mask = _attention_inputs(case, seed)
        n = case["n_kv"]
        # queries enter the scores rounded to f16, as the keys' type asks
        return _attend(q.half().double(), k[:, :n].double(), v[:, :n].double(), None if mask is None else mask.double(),
                       case["D"] ** -0.5)
    return _exact_model(case, seed)


def _exact_model(case: dict, seed: int):
    """The decoder's logits in f64 from the decoded weights (no rounding of activations, K or V)."""
    c = _config(case)
    what = {name: 10 + i for i, (name, _, _) in enumerate(_model_shapes(c))}
    size = {name: (n, k) for name, n, k in _model_shapes(c)}
    prompt, rest = _tokens(case, seed, c.n_vocab)
    P, D = len(prompt), c.head_dim
    S = P + len(rest)

    def product(name, x):
        return _product(x, case["wtype"], *size[name], seed, what[name])

    def norm(x):
        return x / torch.sqrt((x * x).mean(1, keepdim=True) + EPS)

    angle = torch.arange(S, device="cuda", dtype=torch.float64).unsqueeze(1) * c.rope_base ** (
        -2.0 * torch.arange(D // 2, device="cuda", dtype=torch.float64) / D)
    cos, sin = torch.cos(angle).unsqueeze(1), torch.sin(angle).unsqueeze(1)

    def rope(x):
        a, b = x[..., :D // 2], x[..., D // 2:]
        return torch.cat([a * cos - b * sin, a * sin + b * cos], 2)

    ids = torch.tensor(prompt + rest, device="cuda")
    x = _encode(_weight_f32(*size["token_embd"], seed, what["token_embd"])[ids], case["wtype"], values=True)
    mask = torch.full((S, S), -math.inf, device="cuda", dtype=torch.float64).triu(1)
    nq, nk = c.n_head * D, c.n_head_kv * D
    for i in range(c.n_layer):
        qkv = product(f"blk.{i}.attn_qkv", norm(x))
        q = rope(qkv[:, :nq].reshape(S, -1, D)).transpose(0, 1)
        k = rope(qkv[:, nq:nq + nk].reshape(S, -1, D)).transpose(0, 1)
        v = qkv[:, nq + nk:].reshape(S, -1, D).transpose(0, 1)
        a = _attend(q, k, v, mask, D ** -0.5)
        x = x + product(f"blk.{i}.attn_output", a.reshape(S, nq))
        gu = product(f"blk.{i}.ffn_gate_up", norm(x))
        x = x + product(f"blk.{i}.ffn_down", torch.nn.functional.silu(gu[:, :c.n_ff]) * gu[:, c.n_ff:])
    return product("output", norm(x[P - 1:])).cpu().numpy()
