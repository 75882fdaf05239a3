"""The workloads this package is measured on: what a program that serves,
packs or unpacks SE12 weights has it do, called through the public entry
points, over the whole range of sizes and not only at the tuned shapes.

A case is a dict with an "op" and its sizes:

  linear   y = x W^T for one bound matrix (Se12MatVecKernel.multiply), BF16 or
           FP32 activations, 1..32 rows; "tail" = heavy-tailed weights (more
           escapes and raw tiles) instead of Gaussian ones
  grouped  two matrices that share x in one launch (multiply_grouped)
  mlp      the MLP half of a decode step: post-attention norm, gate/up, the
           gate, down_proj (multiply_prenorm + multiply_rowss)
  pack     SE12-encoding a BF16 matrix on the GPU (encode_on_device)
  unpack   the WeightDecoder port on a list of packed matrices, each seen for
           the first time (HipSe12WeightDecoder.decode_to_device)
  embed    an embedding lookup from a packed table (CompressedEmbedding)
  attend   one decode step of attention over a KV cache (se12_step_attention)
  prefill  a whole Gemma-2 prompt pass: logits of the last position
  decode   a whole Gemma-2 decode loop fed with given tokens (a program with
           its own sampler), the step captured in a HIP graph: logits of
           every step

Weights, activations and tokens are drawn on the GPU from the seed alone.
"""

from __future__ import annotations

import math

import torch

from se12_amd import _native as nat
from se12_amd.gemma2 import PROJECTIONS, Gemma2Decoder, Gemma2Shape, Gemma2Weights
from se12_amd.hip import (HipSe12WeightDecoder, Se12MatVecKernel, encode_on_device, multiply_grouped, multiply_prenorm)
from se12_amd.runtime import CompressedEmbedding

TILE_ROWS, TILE_COLS, TILE_BYTES = 16, 256, 6160
EPS = 1e-6


def listed() -> list[dict]:
    return [
        # the smallest call: Gemma-2-2B's down_proj for one new token
        {"name": "down_2b_b1", "op": "linear", "rows": 2304, "cols": 9216, "batch": 1, "x": "bf16", "tail": False},
        # the MLP of one Gemma-2-2B layer for eight sequences' new tokens
        {"name": "mlp_2b_b8", "op": "mlp", "hidden": 2304, "inter": 9216, "batch": 8},
        # gate and up of Gemma-2-9B for sixteen sequences, one launch
        {"name": "gate_up_9b_b16", "op": "grouped", "rows": 14336, "cols": 3584, "batch": 16, "x": "bf16", "tail": False},
        # the tied LM head, heavy-tailed weights, four sequences
        {"name": "lm_head_2b_b4", "op": "linear", "rows": 256000, "cols": 2304, "batch": 4, "x": "bf16", "tail": True},
        # FP32 activations (a model kept in FP32 around packed weights)
        {"name": "down_9b_f32_b8", "op": "linear", "rows": 3584, "cols": 14336, "batch": 8, "x": "f32", "tail": False},
        # a matrix that is no whole number of tiles either way
        {"name": "ragged_b6", "op": "linear", "rows": 5003, "cols": 2887, "batch": 6, "x": "bf16", "tail": False},
        # packing a model: one gate projection
        {"name": "pack_gate_2b", "op": "pack", "rows": 9216, "cols": 2304, "tail": False},
        # restoring BF16 weights from a packed file: gate and up
        {"name": "unpack_2b", "op": "unpack", "rows": 9216, "cols": 2304, "count": 2, "tail": False},
        # the embedding of a 2,048-token prompt
        {"name": "embed_2048", "op": "embed", "rows": 256000, "cols": 2304, "tokens": 2048},
        # attention of Gemma-2-9B for eight sequences, 3,000 tokens into a
        # cache of 8,192
        {"name": "attend_9b_b8", "op": "attend", "batch": 8, "heads": 16, "kv_heads": 8, "head_dim": 256, "max_len": 8192,
         "pos": 3000, "window": 0},
        # a whole prompt through Gemma-2-2B
        {"name": "prefill_2b_1024", "op": "prefill", "layers": 26, "hidden": 2304, "inter": 9216, "heads": 8, "kv_heads": 4,
         "head_dim": 256, "vocab": 256000, "window": 4096, "batch": 1, "prompt": 1024},
        # four tokens through Gemma-2-2B after a 512-token prompt
        {"name": "decode_2b", "op": "decode", "layers": 26, "hidden": 2304, "inter": 9216, "heads": 8, "kv_heads": 4,
         "head_dim": 256, "vocab": 256000, "window": 4096, "batch": 1, "prompt": 512, "steps": 4},
    ]


# ---------------------------------------------------------------------------
# drawn cases
# ---------------------------------------------------------------------------


def _log(rng, lo: float, hi: float) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _dim(rng, lo: int, hi: int) -> int:
    """A matrix dimension: a multiple of 256 (most models), else any size."""
    n = _log(rng, lo, hi)
    return max(256, n // 256 * 256) if rng.random() < 0.65 else n


def _model(rng) -> dict:
    kv = rng.choice([1, 2, 4, 8])
    g = rng.choice([1, 2, 4, 8])
    d = rng.choice([64, 128, 256])
    hidden = 256 * _log(rng, 2, 14)
    return {"layers": rng.randint(1, 4), "hidden": hidden, "inter": 256 * _log(rng, 2, 4 * hidden // 256),
            "heads": kv * g, "kv_heads": kv, "head_dim": d, "vocab": _log(rng, 2000, 64000),
            "window": rng.choice([4096, 4096, 256])}


def draw(rng) -> dict:
    op = rng.choice(["linear"] * 4 + ["grouped"] * 2 + ["mlp", "pack", "pack", "unpack", "embed", "attend", "attend",
                                                         "prefill", "decode"])
    tail = rng.random() < 0.3
    if op in ("linear", "grouped"):
        rows, cols = _dim(rng, 256, 256000 if op == "linear" else 40000), _dim(rng, 256, 16384)
        while rows * cols > (600e6 if op == "linear" else 200e6):
            rows = max(256, rows // 2)
        return {"op": op, "rows": rows, "cols": cols, "batch": _log(rng, 1, 32.49), "x": "f32" if rng.random() < 0.25 else "bf16",
                "tail": tail}
    if op == "mlp":
        hidden = 256 * _log(rng, 4, 20)
        return {"op": op, "hidden": hidden, "inter": 256 * _log(rng, 8, 80), "batch": _log(rng, 1, 32.49)}
    if op == "pack":
        rows, cols = _dim(rng, 256, 64000), _dim(rng, 256, 16384)
        while rows * cols > 200e6:
            rows = max(256, rows // 2)
        return {"op": op, "rows": rows, "cols": cols, "tail": tail}
    if op == "unpack":
        rows, cols = _dim(rng, 256, 40000), _dim(rng, 256, 16384)
        while rows * cols > 100e6:
            rows = max(256, rows // 2)
        return {"op": op, "rows": rows, "cols": cols, "count": rng.randint(2, 4), "tail": tail}
    if op == "embed":
        return {"op": op, "rows": _log(rng, 2000, 64000), "cols": _dim(rng, 256, 5120), "tokens": _log(rng, 1, 8192)}
    if op == "attend":
        max_len = 8 * _log(rng, 16, 2048)
        kv = rng.choice([1, 2, 4, 8])
        batch = _log(rng, 1, 32.49)
        while batch * kv * max_len > 8 * 8 * 8192:
            batch = max(1, batch // 2)
            if batch == 1:
                break
        return {"op": op, "batch": batch, "heads": kv * rng.choice([1, 2, 4, 8]), "kv_heads": kv,
                "head_dim": rng.choice([64, 128, 256]), "max_len": max_len, "pos": rng.randrange(max_len // 16, max_len),
                "window": rng.choice([0, 0, 1024, 4096])}
    m = _model(rng)
    if op == "prefill":
        batch = _log(rng, 1, 8.49)
        return {"op": op, **m, "batch": batch, "prompt": _log(rng, 5, 2048 / batch)}
    return {"op": op, **m, "batch": _log(rng, 1, 32.49), "prompt": _log(rng, 5, 256), "steps": rng.randint(2, 6)}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

DEV = "cuda"


def _gen(seed: int, salt: int) -> torch.Generator:
    g = torch.Generator(device=DEV)
    g.manual_seed((seed * 1_000_003 + salt) % (1 << 62))
    return g


def _weights(rows: int, cols: int, seed: int, salt: int, tail: bool) -> torch.Tensor:
    """BF16 N(0, 0.02); `tail`: Student-t (3 degrees) of that spread with 0.1%
    of the weights at +-8 sigma."""
    g = _gen(seed, salt)
    w = torch.randn((rows, cols), generator=g, device=DEV)
    if not tail:
        return (w * 0.02).to(torch.bfloat16)
    chi2 = torch.zeros_like(w)
    z = torch.empty_like(w)
    for _ in range(3):
        z.normal_(generator=g)
        chi2.addcmul_(z, z)
    w.mul_(torch.rsqrt(chi2.div_(3.0))).mul_(0.02 / math.sqrt(3.0))
    n = max(1, w.numel() // 1000)
    at = torch.randint(0, w.numel(), (n,), generator=g, device=DEV)
    w.view(-1)[at] = (at & 1).float() * 0.32 - 0.16  # by index: one drawn twice gets one value
    return w.to(torch.bfloat16)


def _acts(case: dict, batch: int, cols: int, seed: int, salt: int = 1) -> torch.Tensor:
    x = torch.randn((batch, cols), generator=_gen(seed, salt), device=DEV)
    return x if case.get("x") == "f32" else x.to(torch.bfloat16)


def _mlp_inputs(case: dict, seed: int) -> dict:
    h, b = case["hidden"], case["batch"]
    g = _gen(seed, 50)

    def bf16(*shape, std=1.0):
        return (torch.randn(shape, generator=g, device=DEV) * std).to(torch.bfloat16)

    y_prev = torch.randn((b, h), generator=g, device=DEV)
    # the row sums that the o_proj product writes beside its output
    sq = y_prev.to(torch.bfloat16).float().square()
    return {"y_prev": y_prev, "ss": sq.view(b, h // TILE_ROWS, TILE_ROWS).sum(-1).contiguous(),
            "w1": bf16(h, std=0.1), "w2": bf16(h, std=0.1), "res": bf16(b, h)}


def _attend_inputs(case: dict, seed: int) -> dict:
    b, kv, d, n = case["batch"], case["kv_heads"], case["head_dim"], case["max_len"]
    g = _gen(seed, 60)
    kt = torch.empty((b, kv, d, n), dtype=torch.bfloat16, device=DEV).normal_(generator=g)
    v = torch.empty((b, kv, n, d), dtype=torch.bfloat16, device=DEV).normal_(generator=g)
    qkv = [torch.randn((b, c * d), generator=g, device=DEV) for c in (case["heads"], kv, kv)]
    inv = 1.0 / (10000.0 ** (torch.arange(0, d, 2, dtype=torch.int64, device=DEV).float() / d))
    return {"kt": kt, "v": v, "qkv": qkv, "inv": inv}


def _shape(case: dict) -> Gemma2Shape:
    return Gemma2Shape(layers=case["layers"], hidden=case["hidden"], intermediate=case["inter"], heads=case["heads"],
                       kv_heads=case["kv_heads"], head_dim=case["head_dim"], vocab=case["vocab"],
                       query_pre_attn_scalar=float(case["head_dim"]), sliding_window=case["window"])


def _model_inputs(case: dict, seed: int) -> tuple[Gemma2Weights, torch.Tensor]:
    w = Gemma2Weights.random(_shape(case), torch.device(DEV, torch.cuda.current_device()), seed=seed % 1_000_003)
    g = _gen(seed, 70)
    for lw in w.layers:
        for nm in ("input_norm", "post_attn_norm", "pre_ffw_norm", "post_ffw_norm"):
            lw[nm].normal_(0.0, 0.1, generator=g)
    n = case["prompt"] + case.get("steps", 0)
    return w, torch.randint(0, case["vocab"], (case["batch"], n), generator=g, device=DEV)


def prepare(case: dict, seed: int) -> dict:
    op = case["op"]
    st: dict = {"op": op}
    if op in ("linear", "grouped"):
        n = 2 if op == "grouped" else 1
        st["kernels"] = [Se12MatVecKernel(encode_on_device(_weights(case["rows"], case["cols"], seed, 10 + i, case["tail"])))
                         for i in range(n)]
        st["x"] = _acts(case, case["batch"], case["cols"], seed)
    elif op == "mlp":
        h, n, b = case["hidden"], case["inter"], case["batch"]
        st["gate_up"] = [Se12MatVecKernel(encode_on_device(_weights(n, h, seed, 20 + i, False))) for i in range(2)]
        st["down"] = Se12MatVecKernel(encode_on_device(_weights(h, n, seed, 22, False)))
        st.update(_mlp_inputs(case, seed))
        st["res_out"], st["h"] = torch.empty_like(st["res"]), torch.empty_like(st["res"])
        st["m"] = torch.empty((b, n), dtype=torch.bfloat16, device=DEV)
        st["gu"] = [torch.empty((b, n), dtype=torch.float32, device=DEV) for _ in range(2)]
        st["out"] = torch.empty((b, h), dtype=torch.float32, device=DEV)
        st["out_ss"] = torch.empty((b, h // TILE_ROWS), dtype=torch.float32, device=DEV)
    elif op == "pack":
        st["w"] = _weights(case["rows"], case["cols"], seed, 10, case["tail"])
    elif op == "unpack":
        st["decoder"] = HipSe12WeightDecoder()
        st["tensors"] = [encode_on_device(_weights(case["rows"], case["cols"], seed, 10 + i, case["tail"]))
                         for i in range(case["count"])]
    elif op == "embed":
        k = Se12MatVecKernel(encode_on_device(_weights(case["rows"], case["cols"], seed, 10, False)))
        st["embedding"] = CompressedEmbedding(k, scale=float(case["cols"]) ** 0.5)
        st["ids"] = torch.randint(0, case["rows"], (1, case["tokens"]), generator=_gen(seed, 2), device=DEV)
    elif op == "attend":
        st.update(_attend_inputs(case, seed))
        st["pos"] = torch.tensor(case["pos"], dtype=torch.int64, device=DEV)
        st["out"] = torch.empty((case["batch"], case["heads"] * case["head_dim"]), dtype=torch.bfloat16, device=DEV)
        n = nat.lib().se12_step_attention_workspace(case["batch"], case["heads"], case["kv_heads"], case["head_dim"],
                                                    case["max_len"])
        nat.step_check(min(n, 0))
        st["ws"] = torch.zeros(n, dtype=torch.uint8, device=DEV)
        st["case"] = case
    else:
        w, st["tokens"] = _model_inputs(case, seed)
        encoded = {(li, n): encode_on_device(lw[n]) for li, lw in enumerate(w.layers) for n in PROJECTIONS}
        encoded["embed"] = encode_on_device(w.embed)
        st["decoder"] = Gemma2Decoder(w, "se12", case["batch"], max_len=case["prompt"] + case.get("steps", 0) + 8,
                                      encoded=encoded)
        st["prompt"] = case["prompt"]
        if op == "decode":
            st["decoder"].prefill(st["tokens"][:, :case["prompt"]])
            st["decoder"].capture()
            st["forced"] = [st["tokens"][:, case["prompt"] + i].contiguous() for i in range(case["steps"])]
    return st


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------


@torch.no_grad()
def run(st: dict):
    op = st["op"]
    if op == "linear":
        return st["kernels"][0].multiply(st["x"])
    if op == "grouped":
        return multiply_grouped(st["kernels"], st["x"])
    if op == "mlp":
        multiply_prenorm(st["gate_up"], st["y_prev"], st["w1"], st["w2"], st["res"], st["res_out"], st["h"], EPS,
                         ys=st["gu"], gelu_out=st["m"], y_prev_ss=st["ss"])
        st["down"].multiply_rowss(st["m"], st["out_ss"], y=st["out"])
        return {"residual": st["res_out"], "h": st["h"], "m": st["m"], "out": st["out"], "out_ss": st["out_ss"]}
    if op == "pack":
        t = encode_on_device(st["w"])
        return {"sm": t.sm, "ec": t.ec, "esc": t.esc, "bitmap": t.fallback_bitmap, "raw": t.fallback_raw,
                "codebook": t.codebook}
    if op == "unpack":
        return [st["decoder"].decode_to_device(t) for t in st["tensors"]]
    if op == "embed":
        return st["embedding"](st["ids"])
    if op == "attend":
        c, (q, k, v) = st["case"], st["qkv"]
        nat.step_check(nat.lib().se12_step_attention(
            nat.ptr(q), nat.ptr(k), nat.ptr(v), nat.STEP_F32, q.shape[1], k.shape[1], nat.ptr(st["kt"]), nat.ptr(st["v"]),
            nat.ptr(st["inv"]), nat.ptr(st["pos"]), nat.ptr(st["out"]), c["batch"], c["heads"], c["kv_heads"],
            c["head_dim"], c["max_len"], float(c["head_dim"]) ** -0.5, 50.0, c["window"], nat.ptr(st["ws"]),
            st["ws"].numel(), nat.stream_ptr()))
        return {"out": st["out"], "k_slot": st["kt"][..., c["pos"]], "v_slot": st["v"][:, :, c["pos"]]}
    d = st["decoder"]
    if op == "prefill":
        d.prefill(st["tokens"])
        return d.last_logits
    d.pos.fill_(st["prompt"])
    d.step_index.fill_(1)
    out = []
    for t in st["forced"]:
        d.ids.copy_(t)
        d.decode(1)
        out.append(d.last_logits.clone())
    return torch.stack(out)


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------


def _se12_bytes(rows: int, cols: int) -> int:
    t = -(-rows // TILE_ROWS) * -(-cols // TILE_COLS)
    return t * TILE_BYTES + -(-t // 8) + 15


def _proj_shapes(c: dict) -> list[tuple[int, int]]:
    q, kv = c["heads"] * c["head_dim"], c["kv_heads"] * c["head_dim"]
    h, n = c["hidden"], c["inter"]
    return [(q, h), (kv, h), (kv, h), (h, q), (n, h), (n, h), (h, n)]


def work(case: dict) -> dict:
    op = case["op"]
    if op in ("linear", "grouped"):
        n = 2 if op == "grouped" else 1
        r, k, b = case["rows"], case["cols"], case["batch"]
        return {"bytes": n * (_se12_bytes(r, k) + 4 * b * r) + b * k * (4 if case["x"] == "f32" else 2),
                "flops": 2.0 * n * r * k * b}
    if op == "mlp":
        h, n, b = case["hidden"], case["inter"], case["batch"]
        # the products' FP32 outputs and the MLP's activations are results
        return {"bytes": 2 * _se12_bytes(n, h) + _se12_bytes(h, n) + 4 * h + b * (4 * h + 2 * h + 4 * h // 16)
                + b * (2 * h + 2 * h + 2 * 4 * n + 2 * n + 4 * h + 4 * h // 16), "flops": 6.0 * h * n * b}
    if op == "pack":
        return {"bytes": 2 * case["rows"] * case["cols"] + _se12_bytes(case["rows"], case["cols"]), "flops": 0}
    if op == "unpack":
        return {"bytes": case["count"] * (2 * case["rows"] * case["cols"] + _se12_bytes(case["rows"], case["cols"])),
                "flops": 0}
    if op == "embed":
        return {"bytes": case["tokens"] * (8 + int(3.5 * case["cols"])), "flops": 0}
    if op == "attend":
        b, h, kv, d = case["batch"], case["heads"], case["kv_heads"], case["head_dim"]
        lo = max(0, case["pos"] - case["window"] + 1) if case["window"] else 0
        n = case["pos"] + 1 - lo
        return {"bytes": b * (4 * d * (h + 2 * kv) + 2 * 2 * kv * d * n + 2 * h * d), "flops": 4.0 * b * h * d * n}
    b, t = case["batch"], case["prompt"]
    proj = _proj_shapes(case)
    weights = case["layers"] * sum(_se12_bytes(r, k) for r, k in proj)
    macs = case["layers"] * sum(r * k for r, k in proj)
    head, vh = _se12_bytes(case["vocab"], case["hidden"]), case["vocab"] * case["hidden"]
    kv = 4 * case["layers"] * case["kv_heads"] * case["head_dim"]  # K and V of one position, BF16
    att = 2.0 * case["layers"] * case["heads"] * case["head_dim"]
    if op == "prefill":
        return {"bytes": weights + head + b * t * (8 + int(1.5 * case["hidden"]) + kv) + 2 * b * case["vocab"],
                "flops": 2.0 * b * t * macs + att * b * t * (t + 1) + 2.0 * b * vh}
    n = case["steps"]
    return {"bytes": n * (weights + head + b * (kv * (t + (n + 1) / 2) + 2 * case["vocab"])),
            "flops": 2.0 * n * b * (macs + vh) + 2 * att * b * sum(t + i + 1 for i in range(n))}


def tolerance(case: dict):
    op = case["op"]
    if op in ("pack", "unpack", "embed"):
        return "exact"
    if op in ("linear", "grouped"):   # FP32 sums: 0.7e-7 to 4e-7 off 64 bits
        return {"rel": 2e-6, "max": 2e-5}
    if op == "mlp":                   # BF16 activations between the products: 5e-3 off 64 bits
        return {"rel": 1.5e-2, "max": 1.5e-1}
    if op == "attend":                # scores rounded to BF16: 7e-3 off 64 bits
        return {"rel": 2e-2, "max": 2e-1}
    return {"rel": 3e-2, "max": 3e-1}  # a whole model in BF16: 1.8e-2 off 64 bits


# ---------------------------------------------------------------------------
# the same results in 64 bits, without this package's code
# ---------------------------------------------------------------------------


def _linear64(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """x [B, K] against W [N, K] in 64 bits, in slices of rows of W."""
    step = max(1, (1 << 28) // w.shape[1])
    return torch.cat([x @ w[i:i + step].double().t().contiguous() for i in range(0, w.shape[0], step)], dim=1)


def _norm64(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * (1.0 + w.double())


def _gelu64(x: torch.Tensor) -> torch.Tensor:
    return 0.5 * x * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (x + 0.044715 * x ** 3)))


def _rope64(x: torch.Tensor, pos: torch.Tensor) -> torch.Tensor:
    """x [..., T, d] rotated at positions pos [T]."""
    d = x.shape[-1]
    inv = 1.0 / (10000.0 ** (torch.arange(0, d, 2, dtype=torch.float64, device=x.device) / d))
    f = pos.double()[:, None] * inv
    f = torch.cat((f, f), dim=-1)
    rot = torch.cat((-x[..., d // 2:], x[..., :d // 2]), dim=-1)
    return x * f.cos() + rot * f.sin()


def _softcap64(s: torch.Tensor, cap: float) -> torch.Tensor:
    return torch.tanh(s / cap) * cap


def _model64(case: dict, seed: int) -> torch.Tensor:
    """Logits [B, T, vocab] of the last 1 (prefill) or `steps` positions."""
    w, tokens = _model_inputs(case, seed)
    s = w.shape
    b, t = tokens.shape
    h, kvh, d = s.heads, s.kv_heads, s.head_dim
    g = h // kvh
    x = w.embed[tokens].double() * math.sqrt(s.hidden)
    pos = torch.arange(t, device=DEV)
    back = pos[:, None] - pos[None, :]

    def lin(a, m):
        return _linear64(a.reshape(b * t, -1), m).view(b, t, -1)

    for li, lw in enumerate(w.layers):
        a = _norm64(x, lw["input_norm"])
        q = _rope64(lin(a, lw["q"]).view(b, t, h, d).transpose(1, 2), pos)
        k = _rope64(lin(a, lw["k"]).view(b, t, kvh, d).transpose(1, 2), pos)
        v = lin(a, lw["v"]).view(b, t, kvh, d).transpose(1, 2)
        ok = back >= 0 if li % 2 else (back >= 0) & (back < s.sliding_window)
        o = torch.empty((b, h, t, d), dtype=torch.float64, device=DEV)
        for bi in range(b):
            for hi in range(h):
                kk, vv = k[bi, hi // g], v[bi, hi // g]
                sc = _softcap64(q[bi, hi] @ kk.t().contiguous() * s.query_pre_attn_scalar ** -0.5, s.attn_softcap)
                o[bi, hi] = torch.softmax(sc.masked_fill(~ok, float("-inf")), -1) @ vv.contiguous()
        x = x + _norm64(lin(o.transpose(1, 2).reshape(b, t, h * d), lw["o"]), lw["post_attn_norm"])
        a = _norm64(x, lw["pre_ffw_norm"])
        m = _gelu64(lin(a, lw["gate"])) * lin(a, lw["up"])
        x = x + _norm64(lin(m, lw["down"]), lw["post_ffw_norm"])
    n = case.get("steps", 0) or 1
    x = _norm64(x[:, t - n:], w.final_norm).reshape(b * n, -1)
    return _softcap64(_linear64(x, w.embed), s.final_softcap).view(b, n, s.vocab)


@torch.no_grad()
def exact(case: dict, seed: int):
    op = case["op"]
    if op in ("linear", "grouped"):
        x = _acts(case, case["batch"], case["cols"], seed).double()
        ys = [_linear64(x, _weights(case["rows"], case["cols"], seed, 10 + i, case["tail"]))
              for i in range(2 if op == "grouped" else 1)]
        return ys if op == "grouped" else ys[0]
    if op == "mlp":
        h, n, b = case["hidden"], case["inter"], case["batch"]
        i = _mlp_inputs(case, seed)
        r = i["res"].double() + _norm64(i["y_prev"].double(), i["w1"])
        a = _norm64(r, i["w2"])
        m = _gelu64(_linear64(a, _weights(n, h, seed, 20, False))) * _linear64(a, _weights(n, h, seed, 21, False))
        out = _linear64(m, _weights(h, n, seed, 22, False))
        return {"residual": r, "h": a, "m": m, "out": out,
                "out_ss": out.square().view(b, h // TILE_ROWS, TILE_ROWS).sum(-1)}
    if op == "unpack":
        return [_weights(case["rows"], case["cols"], seed, 10 + i, case["tail"]) for i in range(case["count"])]
    if op == "embed":
        ids = torch.randint(0, case["rows"], (1, case["tokens"]), generator=_gen(seed, 2), device=DEV)
        return _weights(case["rows"], case["cols"], seed, 10, False)[ids].double() * math.sqrt(case["cols"])
    if op == "attend":
        i, p = _attend_inputs(case, seed), case["pos"]
        b, h, kvh, d = case["batch"], case["heads"], case["kv_heads"], case["head_dim"]
        at = torch.tensor([p], device=DEV)
        q = _rope64(i["qkv"][0].double().view(b, h, 1, d), at)
        k = _rope64(i["qkv"][1].double().view(b, kvh, 1, d), at)
        v = i["qkv"][2].double().view(b, kvh, 1, d)
        lo = max(0, p - case["window"] + 1) if case["window"] else 0
        out = torch.empty((b, h, d), dtype=torch.float64, device=DEV)
        for bi in range(b):
            for hi in range(h):
                kv = hi // (h // kvh)
                keys = torch.cat((i["kt"][bi, kv, :, lo:p].double(), k[bi, kv].t()), dim=1).contiguous()
                vals = torch.cat((i["v"][bi, kv, lo:p].double(), v[bi, kv]), dim=0)
                sc = _softcap64(q[bi, hi] @ keys * d ** -0.5, 50.0)
                out[bi, hi] = (torch.softmax(sc, -1) @ vals)[0]
        return {"out": out.view(b, h * d), "k_slot": k.squeeze(2), "v_slot": v.squeeze(2)}
    if op == "prefill":
        return _model64(case, seed)[:, 0]
    if op == "decode":
        return _model64(case, seed).transpose(0, 1).contiguous()
    return None
