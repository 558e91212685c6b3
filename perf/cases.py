"""The work whose time is measured, as a user's program has this package do it, through its public entry points.

Five kinds of call, each over the sizes that it meets in use:

  gemv    one ternary projection of one int8 vector (VelurexHipLayer): tensors on the GPU (``gemv_i32``,
          ``gemv_f32``) or host arrays (``forward``, the drop-in call of a host runtime)
  plan    the projections of one token in one launch (``Plan``), with the int8 inputs staged in every run or ahead
  gemm    one projection of many tokens (``vx_gemm_i32_dev``)
  q2      block-scaled (Q2_0 x Q8_0) projections: one (``Q2Matrix.gemv_f32``) or a token's (``Q2Plan``)
  model   a whole model: a prompt (``Decoder.prefill``), single steps at a context (``Decoder.step``), greedy
          generation (``Decoder.generate``)

Weights are i.i.d. trits with P(-1) = P(+1) = 0.35, activations the absmax int8 codes of N(0, 1) values (the
per-token quantizer's), model weights random with the distributions of the benchmark's models. The package's results
are bit-identical to its reference's by contract, floating point included, so every tolerance is "exact".
"""
import ctypes
import math

import numpy as np
import torch

from quintrit_amd import VelurexHipLayer, _lib
from quintrit_amd.decoder import Decoder, DecoderConfig

RADIX = (1, 3, 9, 28, 84)  # a byte is d0 + 3 d1 + 9 d2 + 28 d3 + 84 d4, each digit a trit + 1
WEIGHT_SCALE = 0.02
NORM_LENGTHS = ("hidden", "qd", "hidden", "ffn")  # attention norm, its sub-norm, FFN norm, its sub-norm

FALCON3_10B = {"family": "falcon3", "hidden": 3072, "heads": 12, "kv_heads": 4, "head_dim": 256, "ffn": 23040}
BITNET_2B = {"family": "bitnet", "hidden": 2560, "heads": 20, "kv_heads": 5, "head_dim": 128, "ffn": 6912}


def listed():
    return [
        # The smallest call: the K or V projection of a small model, one vector, everything on the GPU. Latency only.
        {"name": "gemv_smallest", "kind": "gemv", "rows": 640, "cols": 2560, "entry": "f32"},
        # The widest projection that a program calls on its own (an FFN gate or up of the 10B shapes).
        {"name": "gemv_widest", "kind": "gemv", "rows": 23040, "cols": 3072, "entry": "f32"},
        # The drop-in call of a host runtime: activations and outputs in host arrays (a q or o projection).
        {"name": "forward_host", "kind": "gemv", "rows": 3072, "cols": 3072, "entry": "host"},
        # All projections of one token of the 10B shapes, inputs given as int8: the weight stream of a decode step.
        {"name": "plan_token", "kind": "plan", "layers": 40, "hidden": 3072, "qd": 3072, "kvd": 1024, "ffn": 23040, "raw": True},
        # A small batch of tokens (speculative or batched decoding) on the FFN's down projection.
        {"name": "gemm_batch_8", "kind": "gemm", "rows": 3072, "cols": 23040, "m": 8},
        # An odd number of tokens on odd sizes: no row of the input is aligned, every edge is ragged.
        {"name": "gemm_ragged", "kind": "gemm", "rows": 6913, "cols": 2563, "m": 100},
        # A prefill pass' widest product: 512 tokens on an FFN gate or up of the 10B shapes.
        {"name": "gemm_512", "kind": "gemm", "rows": 23040, "cols": 3072, "m": 512},
        # One block-scaled projection on its own (a q or o projection of the 8B-like shapes).
        {"name": "q2_single", "kind": "q2", "layers": 0, "rows": 4096, "cols": 4096},
        # The block-scaled projections of a token of a small model of the 8B-like layers.
        {"name": "q2_token", "kind": "q2", "layers": 6, "hidden": 4096, "qd": 4096, "kvd": 1024, "ffn": 12288},
        # A chat turn: a short prompt, then greedy tokens one by one (10 of the 10B model's layers, a quarter of its head).
        dict(FALCON3_10B, name="generate", kind="model", layers=10, vocab=32768, ctx=64, new=48, mode="generate"),
        # Steps deep in a context, the host choosing each token from the logits.
        dict(FALCON3_10B, name="steps_long", kind="model", layers=10, vocab=32768, ctx=3900, new=8, mode="steps"),
        # A long prompt of a whole small model: several passes of 512 tokens, attention over the growing context.
        dict(BITNET_2B, name="prefill", kind="model", layers=30, vocab=32064, ctx=1500, new=0, mode="prefill"),
    ]


def draw(rng):
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(("gemv", "gemv", "plan", "gemm", "gemm", "q2", "model", "model"))
    if kind == "gemv":
        return {"kind": kind, "rows": log(64, 23040), "cols": log(160, 23040) // (5 if rng.random() < 0.2 else 1) + 1,
                "entry": rng.choice(("i32", "f32", "host"))}
    if kind == "plan":
        hidden = 64 * log(8, 48)
        return {"kind": kind, "layers": rng.randint(1, 30), "hidden": hidden, "qd": hidden, "kvd": 64 * log(2, 16),
                "ffn": 4 * log(400, 5760), "raw": rng.random() < 0.5}
    if kind == "gemm":
        cols = log(256, 23040)
        return {"kind": kind, "rows": log(256, min(23040, 23040 * 3072 // cols)), "cols": cols, "m": log(2, 512)}
    if kind == "q2":
        if rng.random() < 0.5:
            return {"kind": kind, "layers": 0, "rows": log(64, 12288), "cols": 64 * log(4, 192)}
        return {"kind": kind, "layers": rng.randint(1, 6), "hidden": 64 * log(8, 64), "qd": 64 * log(8, 64),
                "kvd": 64 * log(2, 16), "ffn": 64 * log(16, 192)}
    family = rng.choice(("falcon3", "bitnet"))
    head_dim = rng.choice((64, 128, 256))
    kv_heads, group = rng.randint(1, 5), rng.randint(1, 4)
    mode = rng.choice(("generate", "steps", "prefill"))
    ctx = log(1, 2000) if mode != "generate" else log(1, 300)
    return {"kind": kind, "family": family, "hidden": 32 * log(16, 96), "heads": kv_heads * group, "kv_heads": kv_heads,
            "head_dim": head_dim, "ffn": 4 * log(256, 1728 if family == "bitnet" else 5760), "layers": rng.randint(1, 4),
            "vocab": log(1000, 32768), "ctx": ctx, "new": 0 if mode == "prefill" else rng.randint(2, 8), "mode": mode}


# ---- inputs -------------------------------------------------------------------------------------------------------------


def generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def byte_table():
    """65536 planar bytes with the distribution of five i.i.d. trits."""
    p = np.array([0.35, 0.30, 0.35])
    d = np.stack(np.meshgrid(*[np.arange(3)] * 5, indexing="ij"), -1).reshape(-1, 5)
    cdf = np.cumsum(np.prod(p[d], axis=1))
    at = np.minimum(np.searchsorted(cdf, (np.arange(65536) + 0.5) / 65536.0), len(d) - 1)
    return torch.from_numpy((d @ np.array(RADIX)).astype(np.uint8)[at]).cuda()


def digit_table():
    """Per byte its five digits (rows of bytes that encode nothing hold ones: zero trits)."""
    t = np.ones((256, 5), np.uint8)
    for d in np.stack(np.meshgrid(*[np.arange(3)] * 5, indexing="ij"), -1).reshape(-1, 5):
        t[int(d @ np.array(RADIX))] = d
    return torch.from_numpy(t).cuda()


def planar(g, table, rows, cols):
    """Planar bytes (32 per row and 160 columns: byte j holds columns j, j + 32, ... of its block), zero trits past cols."""
    nb = (cols + 159) // 160
    out = table[torch.randint(0, 65536, (rows * nb * 32,), dtype=torch.int32, device="cuda", generator=g)].view(rows, nb, 32)
    rem = cols - (nb - 1) * 160
    if rem < 160:
        d = digit_table()[out[:, -1].int()].transpose(1, 2).reshape(rows, 160)  # plane-major: the block's columns
        d[:, rem:] = 1
        radix = torch.tensor(RADIX, dtype=torch.int32, device="cuda").view(1, 5, 1)
        out[:, -1] = (d.view(rows, 5, 32).int() * radix).sum(1).to(torch.uint8)
    return out.reshape(-1)


def trits(bytes_, rows, cols):
    """The weights of planar bytes, rows x cols in 64 bits."""
    nb = (cols + 159) // 160
    d = digit_table()[bytes_.view(rows, nb, 32).int()]  # rows, nb, 32, 5
    return d.permute(0, 1, 3, 2).reshape(rows, nb * 160)[:, :cols].double() - 1.0


def matrix(bytes_, rows, cols, scale):
    h = ctypes.c_void_p()
    _lib.check(_lib.lib().vx_matrix_create_dev(ctypes.c_void_p(bytes_.data_ptr()), bytes_.numel(), rows, cols,
                                               ctypes.c_float(scale), ctypes.byref(h)))
    return VelurexHipLayer._from_handle(h)


def codes(g, m, n):
    """m rows of int8 codes of N(0, 1) values (absmax, 127 levels) and their scales."""
    x = torch.randn(m, n, device="cuda", generator=g)
    s = 127.0 / x.abs().amax(1, keepdim=True)
    return torch.round(x * s).clamp(-128, 127).to(torch.int8), s[:, 0].contiguous()


def token_shapes(case):
    """The projections of a layer as one program launches them: q, k and v of one input, o, gate and up, down."""
    h, q, kv, f = case["hidden"], case["qd"], case["kvd"], case["ffn"]
    return ((q + 2 * kv, h), (h, q), (2 * f, h), (h, f))


def q2_shapes(case):
    if case["layers"] == 0:
        return [(case["rows"], case["cols"])]
    h, q, kv, f = case["hidden"], case["qd"], case["kvd"], case["ffn"]
    return [(q, h), (kv, h), (kv, h), (h, q), (f, h), (f, h), (h, f)] * case["layers"]


def stream():
    return ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)


def spread(g, n):
    """n scales, log-uniform in [0.005, 0.05]."""
    u = torch.rand(n, device="cuda", generator=g)
    return torch.exp(math.log(0.005) + u * (math.log(0.05) - math.log(0.005)))


def q2_inputs(case, seed):
    g, table = generator(seed), byte_table()
    for rows, cols in q2_shapes(case):
        w = planar(g, table, rows, cols)
        yield rows, cols, w, spread(g, rows * cols // 64).half(), codes(g, 1, cols)[0][0], spread(g, cols // 32)


def model_config(case):
    max_ctx = min(8192, (case["ctx"] + case["new"] + 255) // 256 * 256)
    if case["family"] == "falcon3":
        return DecoderConfig.falcon3(case["layers"], case["hidden"], case["heads"], case["kv_heads"], case["head_dim"],
                                     case["ffn"], case["vocab"], max_ctx)
    return DecoderConfig(case["layers"], case["hidden"], case["heads"], case["kv_heads"], case["head_dim"], case["ffn"],
                         case["vocab"], max_ctx)


def model_inputs(case, seed):
    """The model's weights one after the other, as ("proj", layer, kind, bytes), ("norm", layer, kind, values),
    ("emb" or "head", -, -, values), and at last ("tokens", -, -, ids)."""
    cfg, g, table = model_config(case), generator(seed), byte_table()
    lengths = {"hidden": cfg.hidden, "qd": cfg.n_heads * cfg.head_dim, "ffn": cfg.ffn}
    for layer in range(cfg.n_layers):
        for kind in range(7):
            yield "proj", layer, kind, planar(g, table, *cfg.projection_shape(kind))
        for kind in (0, 1, 2, 3) if cfg.has_sub_norms else (0, 2):
            yield "norm", layer, kind, 0.75 + 0.5 * torch.rand(lengths[NORM_LENGTHS[kind]], device="cuda", generator=g)
    yield "norm", cfg.n_layers, 0, 0.75 + 0.5 * torch.rand(cfg.hidden, device="cuda", generator=g)
    for which in ("emb", "head") if cfg.untied else ("emb",):
        t = torch.randn(cfg.vocab * cfg.hidden, device="cuda", generator=g) * 0.02
        yield which, -1, -1, t.to(torch.float16 if cfg.emb_f16 else torch.bfloat16)
    yield "tokens", -1, -1, torch.randint(0, cfg.vocab, (case["ctx"] + case["new"],), device="cuda", generator=g)


# ---- one case -----------------------------------------------------------------------------------------------------------


def prepare(case, seed):
    kind = case["kind"]
    if kind == "gemv":
        rows, cols, g = case["rows"], case["cols"], generator(seed)
        layer = matrix(planar(g, byte_table(), rows, cols), rows, cols, WEIGHT_SCALE)
        q, s = codes(g, 1, cols)
        if case["entry"] == "host":
            return {"case": case, "layer": layer, "x": q[0].cpu().numpy(), "s": float(s[0]), "out": np.empty(rows, np.float32)}
        out = torch.empty(rows, dtype=torch.int32 if case["entry"] == "i32" else torch.float32, device="cuda")
        return {"case": case, "layer": layer, "x": q[0].contiguous(), "s": float(s[0]), "out": out}
    if kind == "plan":
        g, table, keep, jobs = generator(seed), byte_table(), [], []
        shapes = token_shapes(case) * case["layers"]
        out = torch.empty(sum(r for r, _ in shapes), dtype=torch.float32, device="cuda")
        scales, at = torch.empty(len(shapes), device="cuda"), 0
        for i, (rows, cols) in enumerate(shapes):
            layer = matrix(planar(g, table, rows, cols), rows, cols, WEIGHT_SCALE)
            q, s = codes(g, 1, cols)
            scales[i] = s[0]
            n = _lib.staged_bytes(cols)
            staged = torch.empty(n, dtype=torch.uint8, device="cuda")
            if not case["raw"]:
                _lib.check(_lib.lib().vx_stage_acts_dev(ctypes.c_void_p(q.data_ptr()), cols, cols,
                                                        ctypes.c_void_p(staged.data_ptr()), n, stream()))
            keep.append((layer, q, staged))
            jobs.append(_lib.GemvJob(out_f32=1, matrix=layer.handle.value, staged=staged.data_ptr(), staged_len=n,
                                     act_scale_dev=scales.data_ptr() + 4 * i, out=out.data_ptr() + 4 * at,
                                     out_capacity=rows, acts=q.data_ptr() if case["raw"] else None))
            at += rows
        return {"case": case, "plan": _lib.Plan(jobs), "keep": keep, "scales": scales, "out": out}
    if kind == "gemm":
        rows, cols, m, g = case["rows"], case["cols"], case["m"], generator(seed)
        layer = matrix(planar(g, byte_table(), rows, cols), rows, cols, WEIGHT_SCALE)
        n = ctypes.c_size_t()
        _lib.check(_lib.lib().vx_gemm_workspace_bytes(layer.handle, m, ctypes.byref(n)))
        return {"case": case, "layer": layer, "x": codes(g, m, cols)[0],
                "ws": torch.empty(n.value, dtype=torch.uint8, device="cuda"),
                "out": torch.empty(m, rows, dtype=torch.int32, device="cuda")}
    if kind == "q2":
        keep, jobs, at = [], [], 0
        out = torch.empty(sum(r for r, _ in q2_shapes(case)), dtype=torch.float32, device="cuda")
        for rows, cols, w, ws, x, xs in q2_inputs(case, seed):
            m = _lib.Q2Matrix(w.cpu().numpy(), ws.cpu().numpy(), rows, cols)
            keep.append((m, x, xs))
            jobs.append(_lib.Q2Job(matrix=m.handle.value, acts=x.data_ptr(), acts_len=cols, act_scales=xs.data_ptr(),
                                   n_act_scales=cols // 32, out=out.data_ptr() + 4 * at, out_capacity=rows))
            at += rows
        return {"case": case, "keep": keep, "out": out, "plan": _lib.Q2Plan(jobs) if case["layers"] else None}
    cfg = model_config(case)
    dec = Decoder(cfg)
    for what, layer, kind, v in model_inputs(case, seed):
        if what == "proj":
            rows, cols = cfg.projection_shape(kind)
            dec.adopt_projection(layer, kind, matrix(v, rows, cols, 1.0 / math.sqrt(cols)))
        elif what == "norm":
            dec.set_norm(layer, kind, v.cpu().numpy())
        elif what == "tokens":
            tokens = v.cpu().numpy().astype(np.uint32)
        else:
            (dec.set_embedding if what == "emb" else dec.set_head)(v.view(torch.int16).cpu().numpy().view(np.uint16))
    if case["mode"] == "steps":
        dec.prefill(tokens[:case["ctx"]], want_logits=False)
    return {"case": case, "dec": dec, "tokens": tokens}


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "gemv":
        layer, x, out = state["layer"], state["x"], state["out"]
        if case["entry"] == "host":
            layer.forward(x, state["s"], out)
        elif case["entry"] == "i32":
            layer.gemv_i32(x, out)
        else:
            layer.gemv_f32(x, state["s"], out)
        return out
    if kind == "plan":
        state["plan"].run(stream())
        return state["out"]
    if kind == "gemm":
        x, out, ws = state["x"], state["out"], state["ws"]
        _lib.check(_lib.lib().vx_gemm_i32_dev(state["layer"].handle, ctypes.c_void_p(x.data_ptr()), case["m"], case["cols"],
                                              ctypes.c_void_p(out.data_ptr()), case["rows"], ctypes.c_void_p(ws.data_ptr()),
                                              ws.numel(), stream()))
        return out
    if kind == "q2":
        if state["plan"] is not None:
            state["plan"].run(stream())
        else:
            m, x, xs = state["keep"][0]
            m.gemv_f32(x, xs, state["out"], stream())
        return state["out"]
    dec, tokens, ctx, new = state["dec"], state["tokens"], case["ctx"], case["new"]
    if case["mode"] == "prefill":
        return dec.prefill(tokens)
    if case["mode"] == "steps":
        return [dec.step(int(tokens[ctx + i]), ctx + i) for i in range(new)]
    ids = dec.generate(tokens[:ctx], new)
    return {"ids": np.array(ids), "next": dec.step(ids[-1], ctx + new - 1)}


def shapes_of(case):
    """Every (rows, cols) that one token of the case multiplies."""
    if case["kind"] == "plan":
        return list(token_shapes(case)) * case["layers"]
    if case["kind"] == "q2":
        return q2_shapes(case)
    if case["kind"] == "model":
        cfg = model_config(case)
        return [cfg.projection_shape(k) for k in range(7)] * case["layers"]
    return [(case["rows"], case["cols"])]


def work(case):
    weights = sum(r * c for r, c in shapes_of(case))
    vectors = sum(c + 4 * r for r, c in shapes_of(case))  # int8 in, 32 bits out
    if case["kind"] == "q2":
        return {"bytes": weights * (0.2 + 2 / 64) + vectors + sum(c / 8 for _, c in shapes_of(case)), "flops": 2 * weights}
    if case["kind"] != "model":
        m = case.get("m", 1)
        return {"bytes": weights / 5 + m * vectors, "flops": 2 * m * weights}
    cfg = model_config(case)
    qd, kvd = cfg.n_heads * cfg.head_dim, cfg.n_kv_heads * cfg.head_dim
    head, kv_row = cfg.vocab * cfg.hidden, 4 * kvd * cfg.n_layers  # the head's weights; K and V of a position, f16
    first = 0 if case["mode"] == "steps" else case["ctx"]  # positions of the prefill passes
    # prompt: the weights once per pass, K and V written; step: the weights, the head, K and V of the context
    bytes_, flops = 0.0, 0.0
    if first:
        bytes_ += weights / 5 * -(-first // 512) + first * kv_row + 2 * head
        flops += 2 * first * weights + 2 * first * first * qd * cfg.n_layers + 2 * head
    for i in range(case["new"]):
        pos = case["ctx"] + i
        bytes_ += weights / 5 + 2 * head + 4 * cfg.vocab + pos * kv_row
        flops += 2 * weights + 4 * pos * qd * cfg.n_layers + 2 * head
    return {"bytes": bytes_, "flops": flops}


def tolerance(case):
    # Integer sums are exact; every floating operation is done in the reference's order and rounding, so a correct
    # implementation of this package's contract returns the same bits (two runs and the oracle agree bit for bit).
    return "exact"


# ---- the same in 64 bits ------------------------------------------------------------------------------------------------


def exact(case, seed):
    kind = case["kind"]
    if kind == "gemv":
        rows, cols, g = case["rows"], case["cols"], generator(seed)
        w = trits(planar(g, byte_table(), rows, cols), rows, cols)
        q, s = codes(g, 1, cols)
        acc = w @ q[0].double()
        return acc if case["entry"] == "i32" else acc * (WEIGHT_SCALE / float(s[0]))
    if kind == "plan":
        g, table, out = generator(seed), byte_table(), []
        for rows, cols in token_shapes(case) * case["layers"]:
            w = planar(g, table, rows, cols)
            q, s = codes(g, 1, cols)
            out.append(trits(w, rows, cols) @ q[0].double() * (WEIGHT_SCALE / float(s[0])))
        return torch.cat(out)
    if kind == "gemm":
        rows, cols, g = case["rows"], case["cols"], generator(seed)
        w = trits(planar(g, byte_table(), rows, cols), rows, cols)
        return codes(g, case["m"], cols)[0].double() @ w.T
    if kind == "q2":
        out = []
        for rows, cols, w, ws, x, xs in q2_inputs(case, seed):
            t = trits(w, rows, cols) * ws.double().view(rows, cols // 64).repeat_interleave(64, 1)
            out.append(t @ (x.double() * xs.double().repeat_interleave(32)))
        return torch.cat(out)
    if case["mode"] == "generate":  # the tokens that it continues are its own choice
        return None
    logits = model_exact(case, seed)
    if case["mode"] == "prefill":
        return [logits[0], None]
    return [[row, None] for row in logits]


def model_exact(case, seed):
    """Logits of the last position (prefill) or of the case's steps: the model in 64 bits, with its int8 activations."""
    cfg = model_config(case)
    parts = {}
    for what, layer, kind, v in model_inputs(case, seed):
        parts[what, layer, kind] = v
    tokens = parts["tokens", -1, -1]
    if case["mode"] == "prefill":
        tokens = tokens[:case["ctx"]]
    n, hd, half = len(tokens), cfg.head_dim, cfg.head_dim // 2
    emb = parts["emb", -1, -1].view(cfg.vocab, cfg.hidden)
    head = (parts["head", -1, -1] if cfg.untied else parts["emb", -1, -1]).view(cfg.vocab, cfg.hidden)

    def norm(x, layer, kind):
        if ("norm", layer, kind) not in parts:
            return x
        return x / torch.sqrt((x * x).mean(1, keepdim=True) + cfg.rms_eps) * parts["norm", layer, kind].double()

    def product(x, layer, *kinds):
        amax = x.abs().amax(1, keepdim=True)
        s = torch.where(amax > 0, 127.0 / amax, torch.ones_like(amax))
        q, out = torch.floor((x * s).abs() + 0.5).copysign(x), []
        for kind in kinds:
            rows, cols = cfg.projection_shape(kind)
            out.append(q @ trits(parts["proj", layer, kind], rows, cols).T / s / math.sqrt(cols))
        return out

    angle = torch.arange(n, device="cuda").double()[:, None] * cfg.rope_theta ** (
        -2.0 * torch.arange(half, device="cuda").double() / hd)
    cos, sin = angle.cos()[:, None], angle.sin()[:, None]

    def rope(x):
        x = x.view(n, -1, hd)
        a, b = (x[..., 0::2], x[..., 1::2]) if cfg.rope_mode else (x[..., :half], x[..., half:])
        c, d = a * cos - b * sin, a * sin + b * cos
        return torch.stack((c, d), -1).flatten(2) if cfg.rope_mode else torch.cat((c, d), -1)

    mask = torch.ones(n, n, dtype=torch.bool, device="cuda").tril()
    x = emb[tokens].double()
    for layer in range(cfg.n_layers):
        q, k, v = product(norm(x, layer, 0), layer, 0, 1, 2)
        q, k, v = rope(q), rope(k), v.view(n, -1, hd)
        att = torch.empty_like(q)
        for h in range(cfg.n_heads):
            kv = h // (cfg.n_heads // cfg.n_kv_heads)
            p = (q[:, h] @ k[:, kv].T.contiguous() / math.sqrt(hd)).masked_fill(~mask, -math.inf).softmax(1)
            att[:, h] = p @ v[:, kv]
        x = x + product(norm(att.reshape(n, -1), layer, 1), layer, 3)[0]
        gate, up = product(norm(x, layer, 2), layer, 4, 5)
        act = gate * torch.sigmoid(gate) if cfg.act else gate.clamp(min=0) ** 2
        x = x + product(norm(act * up, layer, 3), layer, 6)[0]
    keep = x[-1:] if case["mode"] == "prefill" else x[case["ctx"]:]
    return norm(keep, cfg.n_layers, 0) @ head.double().T
