"""The work that a program has this backend do, as measurable cases.

A case is a step of a transformer trunk that runs through ``tessera_amd.Backend``: the launches that
``Backend.LaunchKernel`` gets, in the order and with the kernel ids that the regime rules of
``tessera_amd/host/project.hpp`` give for the row count, over buffers that the program owns.  Rows are
the tokens of one call: 1 in decode, 2..16 when a draft is verified, more in prefill.

Kinds:
  layer  norm, q/k/v projections, rotary embedding, cache write, attention, output projection, residual,
         then the feed-forward half: one layer as a whole
  attn   the attention half of a layer alone, over a cache of ``context`` earlier positions
  ffn    the feed-forward half alone (gate, up, silu, down, residual)
  moe    routed experts with a shared expert and its gate (one row), or the routed part of a chunk
  head   final norm, output head, top candidates
  proj   one projection in one of the weight formats

Sizes are those of this repository's benchmark and tests (hidden 5120 with 17408; 24 query heads over 4
key heads of 256; 256 experts of 512 over hidden 2048, eight taken) and generic ones.
"""
from __future__ import annotations

import torch

from tessera_amd import CreateBackend, KernelLaunch

#: bytes of 256 weights (MXFP4 and FP8: exclusive of what is stored once a row)
BYTES_256 = {"q4k": 144, "q5k": 176, "q6k": 210, "mxfp4": 136, "fp8": 256}
#: bytes of one key or value element in the cache
BYTES_KV = {"f32": 4.0, "f16": 2.0, "q8": 1.0, "q4": 0.5, "fp8": 1.0}


def listed():
    return [
        # a small model's decode step: fifteen short launches, where each launch's own cost counts
        {"name": "layer_small_decode", "kind": "layer", "rows": 1, "hidden": 1024, "inter": 3072, "heads": 16, "kv_heads": 4,
         "head_dim": 64, "context": 301, "window": 0, "cache": "f16", "weights": "q4k", "v": "q6k", "down": "q6k"},
        # the feed-forward half of one decoded token at the benchmark's size: weights are read once
        {"name": "ffn_q4k_decode", "kind": "ffn", "rows": 1, "hidden": 5120, "inter": 17408, "weights": "q4k", "down": "q4k"},
        # a draft of five tokens verified; half of a Q4_K_M file's down projections are Q6_K
        {"name": "ffn_q4k_verify", "kind": "ffn", "rows": 5, "hidden": 5120, "inter": 17408, "weights": "q4k", "down": "q6k"},
        # a prefill chunk of the same layer
        {"name": "ffn_q4k_prefill", "kind": "ffn", "rows": 2048, "hidden": 5120, "inter": 17408, "weights": "q4k", "down": "q6k"},
        # the MXFP4 checkpoint's decode with a draft of four: activations quantized per token
        {"name": "ffn_mxfp4_verify", "kind": "ffn", "rows": 4, "hidden": 5120, "inter": 17408, "weights": "mxfp4", "down": "mxfp4"},
        # and its prefill of a 453-token prompt, activations in fp32
        {"name": "ffn_mxfp4_prefill", "kind": "ffn", "rows": 453, "hidden": 5120, "inter": 17408, "weights": "mxfp4", "down": "mxfp4"},
        # one token against a long conversation in an int8 cache
        {"name": "attn_decode_long", "kind": "attn", "rows": 1, "hidden": 5120, "heads": 24, "kv_heads": 4, "head_dim": 256,
         "context": 9300, "window": 0, "cache": "q8", "weights": "q4k", "v": "q6k"},
        # a chunk of a long prompt that follows 2000 tokens already in the fp16 cache
        {"name": "attn_prefill", "kind": "attn", "rows": 512, "hidden": 5120, "heads": 24, "kv_heads": 4, "head_dim": 256,
         "context": 2000, "window": 0, "cache": "f16", "weights": "q4k", "v": "q6k"},
        # the routed experts of one decoded token, and of a prefill chunk
        {"name": "moe_decode", "kind": "moe", "rows": 1, "hidden": 2048, "inter": 512, "experts": 256, "top_k": 8},
        {"name": "moe_prefill", "kind": "moe", "rows": 512, "hidden": 2048, "inter": 512, "experts": 256, "top_k": 8},
        # the output head of one decoded token: the largest matrix of a step, and the candidates to sample from
        {"name": "head_decode", "kind": "head", "rows": 1, "hidden": 5120, "vocab": 131072, "weights": "q6k", "top_k": 8},
        # a projection of an FP8 checkpoint in prefill
        {"name": "proj_fp8_prefill", "kind": "proj", "rows": 300, "n": 6144, "k": 5120, "weights": "fp8"},
    ]


def draw(rng):
    def between(lo, hi, step=1):
        """A multiple of `step`, evenly over the logarithm of the range."""
        v = lo * (hi / lo) ** rng.random()
        return max(lo, min(hi, int(round(v / step)) * step))

    def rows(most):
        return rng.choice([1, 1, between(2, 16), between(17, most), between(17, most)])

    kind = rng.choice(["layer", "attn", "attn", "ffn", "ffn", "moe", "head", "proj", "proj"])
    case = {"kind": kind}
    if kind in ("layer", "attn"):
        group, head_dim = rng.choice([1, 2, 3, 4, 6, 8]), rng.choice([64, 96, 128, 256])
        kv_heads = rng.choice([1, 2, 4, 8]) if head_dim <= 128 else rng.choice([1, 2, 4])
        while group * kv_heads * head_dim % 256 != 0 or group * kv_heads * head_dim > 6144:
            group, kv_heads = rng.choice([1, 2, 4, 6, 8]), rng.choice([2, 4, 8])
        most = 512 if kind == "attn" else 256
        case.update(rows=rows(most), hidden=between(768, 5120, 256), heads=group * kv_heads, kv_heads=kv_heads, head_dim=head_dim,
                    context=between(1, 9300), cache=rng.choice(["f16", "f16", "q8", "q8", "f32", "fp8", "q4"]),
                    weights=rng.choice(["q4k", "q4k", "q5k"]), v=rng.choice(["q6k", "q4k"]))
        case["window"] = between(128, 4096) if rng.random() < 0.2 else 0
        if case["rows"] > 16:
            case["context"] = between(1, 2000)
        if kind == "layer":
            case.update(inter=between(2048, 8192, 256), down=rng.choice(["q6k", "q4k"]))
    elif kind == "ffn":
        weights = rng.choice(["q4k", "q4k", "mxfp4", "mxfp4"])
        case.update(rows=rows(2048), hidden=between(1024, 5120, 256), inter=between(2048, 17408, 256), weights=weights,
                    down="mxfp4" if weights == "mxfp4" else rng.choice(["q4k", "q6k"]))
    elif kind == "moe":
        case.update(rows=rows(512), hidden=between(1024, 2048, 256), inter=rng.choice([256, 512, 768]),
                    experts=rng.choice([32, 64, 128, 256]), top_k=rng.choice([2, 4, 6, 8]))
    elif kind == "head":
        case.update(rows=rng.choice([1, 1, 2, 3, 4]), hidden=between(1024, 5120, 256), vocab=between(32000, 131072),
                    weights=rng.choice(["q6k", "q6k", "q4k"]), top_k=rng.choice([1, 2, 4, 8]))
    else:
        weights = rng.choice(["fp8", "fp8", "q5k", "q6k", "q4k", "mxfp4"])
        case.update(rows=rows(300 if weights == "fp8" else 2048), n=between(512, 6144), k=between(1024, 5120, 256), weights=weights)
    return case


# ---- inputs --------------------------------------------------------------------------------------
# Weights of a standard deviation near 0.02 about zero, as a trained layer's: in the K-quants the
# sub-block scales differ and the minimum cancels the quants' mean.

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _bytes(g, *shape):
    return torch.randint(0, 256, shape, dtype=torch.uint8, device="cuda", generator=g)


def _half_bytes(g, blocks, lo, hi):
    v = torch.rand(blocks, device="cuda", generator=g) * (hi - lo) + lo
    return v.half().view(torch.uint8).view(blocks, 2)


def _pack_scales(sc, mn):
    """Eight 6-bit scales and minimums a block -> 12 bytes (the K-quants' packing)."""
    low = (sc[:, :4] & 63) | ((sc[:, 4:] >> 4) << 6)
    mid = (mn[:, :4] & 63) | ((mn[:, 4:] >> 4) << 6)
    return torch.cat([low, mid, (sc[:, 4:] & 15) | ((mn[:, 4:] & 15) << 4)], dim=1)


def _weights(g, kind, n, k):
    """An n x k matrix in the layout of its format; FP8: (codes, one fp32 scale a row)."""
    if kind == "fp8":
        codes = torch.empty(n, k, dtype=torch.uint8, device="cuda")
        scales = torch.empty(n, device="cuda")
        for r in range(0, n, 8192):
            w = torch.randn(min(8192, n - r), k, device="cuda", generator=g) * 0.02
            s = w.abs().amax(1) / 448.0
            scales[r:r + 8192] = s
            codes[r:r + 8192] = (w / s[:, None]).clamp(-448, 448).to(torch.float8_e4m3fn).view(torch.uint8)
        return codes.view(-1), scales
    if kind == "mxfp4":
        scales = torch.randint(127 - 9, 127 - 5, (n * k // 32,), dtype=torch.uint8, device="cuda", generator=g)
        return torch.cat([_bytes(g, n * k // 2), scales])
    nb = n * k // 256
    if kind == "q6k":
        w = _bytes(g, nb, 210)
        sign = torch.randint(0, 2, (nb, 16), dtype=torch.int8, device="cuda", generator=g) * 2 - 1
        w[:, 192:208] = (torch.randint(32, 128, (nb, 16), dtype=torch.int8, device="cuda", generator=g) * sign).view(torch.uint8)
        w[:, 208:210] = _half_bytes(g, nb, 1e-5, 1.8e-5)
        return w.view(-1)
    w = _bytes(g, nb, BYTES_256[kind])
    sc = torch.randint(20, 64, (nb, 8), dtype=torch.uint8, device="cuda", generator=g)
    d = _half_bytes(g, nb, 8e-5, 1.4e-4) if kind == "q4k" else _half_bytes(g, nb, 4e-5, 7e-5)
    w[:, 0:2] = d
    w[:, 2:4] = (d.contiguous().view(torch.float16).float() * (7.5 if kind == "q4k" else 15.5)).half().view(torch.uint8).view(nb, 2)
    w[:, 4:16] = _pack_scales(sc, sc)
    return w.view(-1)


class _Program:
    """The launches of one pass, built once, and the device memory that they use."""

    def __init__(self):
        self.backend = CreateBackend()
        self.steps, self.held, self.out = [], [], {}
        self._kernels = {}

    def wrap(self, t):
        self.held.append(t)
        return self.backend.WrapBuffer(t.data_ptr(), t.numel() * t.element_size())

    def empty(self, *shape, dtype=torch.float32):
        t = torch.empty(shape, dtype=dtype, device="cuda")
        return t, self.wrap(t)

    def call(self, name, buffers, scalars, grid=1):
        if name not in self._kernels:
            self._kernels[name] = self.backend.LoadKernel(name)
        launch = KernelLaunch(grid_x=max(1, int(grid)), buffers=buffers, scalars=scalars)
        self.steps.append((self.backend.LaunchKernel, (self._kernels[name], launch)))

    def copy(self, dst, dst_off, src, nbytes):
        self.steps.append((self.backend.CopyD2D, (dst, dst_off, src, 0, nbytes)))

    # -- one projection: c = a w^T, by the regime rules for the format and the row count --------------
    def project(self, kind, a, w, m, n, k, c=None):
        if c is None:
            c = self.empty(m, n)[1]
        grid = (m * n + 7) // 8
        if kind == "fp8":
            self.call("gemm_fp8", [a, w[0], w[1], c], [m, n, k], (m * n + 255) // 256)
        elif kind == "mxfp4":
            if m <= 16:
                codes, scale = self.empty(m, k, dtype=torch.uint8)[1], self.empty(m)[1]
                self.call("quantize_fp8_pack_rows", [a, codes, scale], [m, k], m)
                self.project_quantized(codes, scale, w, m, n, k, c)
            else:
                self.call("gemm_mxfp4_batched", [a, w[0], c], [m, n, k], grid)
        elif m == 1:
            self.call(f"gemm_{kind}_vec", [a, w[0], c], [m, n, k, 1], grid)
        elif m <= 5:
            self.call(f"gemm_{kind}_rows{m}", [a, w[0], c], [m, n, k, 1], (n + 7) // 8)
        elif kind == "q4k" and m >= 64:
            self.call("gemm_q4k_wmma", [a, w[0], c], [m, n, k], (n + 63) // 64)
        else:
            self.call(f"gemm_{kind}_batched", [a, w[0], c], [m, n, k], grid)
        return c

    def project_quantized(self, codes, scale, w, m, n, k, c):
        self.call("gemm_mxfp4_wmma", [codes, w[0], scale, w[1], c], [m, n, k, 1, 0], n // 16)

    def weights(self, g, kind, n, k):
        w = _weights(g, kind, n, k)
        if kind == "fp8":
            return self.wrap(w[0]), self.wrap(w[1])
        if kind == "mxfp4":
            packed, (_, ref) = self.wrap(w), self.empty(n, dtype=torch.uint8)
            self.backend.LaunchKernel(self.backend.LoadKernel("mxfp4_row_ref"), KernelLaunch(buffers=[packed, ref], scalars=[n, k]))
            return packed, ref
        return (self.wrap(w),)


def _f32_bits(x):
    return int(torch.tensor(x, dtype=torch.float32).view(torch.int32).item()) & 0xFFFFFFFF


def _norm(p, g, x, rows, cols):
    w = p.wrap(torch.rand(cols, device="cuda", generator=g) + 0.5)
    y = p.empty(rows, cols)[1]
    p.call("rmsnorm", [x, w, y], [rows, cols, _f32_bits(1e-6)], rows)
    return y


def _ffn_kind(c):
    """Gate and up are Q4_K also where the attention half holds Q5_K (as K-quant files mix them)."""
    return "mxfp4" if c["weights"] == "mxfp4" else "q4k"


def _ffn(p, g, c, x):
    m, h, f = c["rows"], c["hidden"], c["inter"]
    xn = _norm(p, g, x, m, h)
    kind = _ffn_kind(c)
    gate, up = p.weights(g, kind, f, h), p.weights(g, kind, f, h)
    down = p.weights(g, c["down"], h, f)
    phi, y, (out, dout) = p.empty(m, f)[1], p.empty(m, h)[1], p.empty(m, h)
    if kind == "q4k":
        p.call("ffn_gate_up_silu_q4k", [xn, gate[0], up[0], phi], [m, f, h], (m * f + 7) // 8)
    else:
        a, b = p.empty(m, f)[1], p.empty(m, f)[1]
        if m <= 16:   # one quantization of the rows for both products
            codes, scale = p.empty(m, h, dtype=torch.uint8)[1], p.empty(m)[1]
            p.call("quantize_fp8_pack_rows", [xn, codes, scale], [m, h], m)
            p.project_quantized(codes, scale, gate, m, f, h, a)
            p.project_quantized(codes, scale, up, m, f, h, b)
        else:
            p.project("mxfp4", xn, gate, m, f, h, a)
            p.project("mxfp4", xn, up, m, f, h, b)
        p.call("silu_mul", [a, b, phi], [m * f], (m * f + 255) // 256)
    p.project(c["down"], phi, down, m, h, f, y)
    p.call("add", [x, y, dout], [m * h], (m * h + 255) // 256)
    p.out["hidden"] = out
    return dout


def _cache(g, kind, positions, width):
    """Keys or values of earlier positions as the cache holds them: (elements or codes, scales)."""
    v = torch.randn(positions, width, device="cuda", generator=g)
    if kind == "f32":
        return v, None
    if kind == "f16":
        return v.half(), None
    amax = v.abs().amax(1)
    if kind == "fp8":
        s = amax / 448.0
        return (v / s[:, None]).clamp(-448, 448).to(torch.float8_e4m3fn).view(torch.uint8), s
    s = amax / (127.0 if kind == "q8" else 7.0)
    q = (v / s[:, None]).round().to(torch.int8)
    if kind == "q8":
        return q.view(torch.uint8), s
    q = q.view(torch.uint8) & 15
    return (q[:, 0::2] | (q[:, 1::2] << 4)).contiguous(), s


def _attn(p, g, c, x):
    m, h, heads, kv, d, past, cache, window = (c[n] for n in ("rows", "hidden", "heads", "kv_heads", "head_dim", "context", "cache", "window"))
    width, n = kv * d, past + m
    xn = _norm(p, g, x, m, h)
    wq, wk, wv = p.weights(g, c["weights"], heads * d, h), p.weights(g, c["weights"], width, h), p.weights(g, c["v"], width, h)
    wo = p.weights(g, c["weights"], h, heads * d)
    q = p.project(c["weights"], xn, wq, m, heads * d, h)
    k = p.project(c["weights"], xn, wk, m, width, h)
    v = p.project(c["v"], xn, wv, m, width, h)
    theta = _f32_bits(1e6)
    p.call("rope", [q], [m, heads, d, d, past, theta], (m * heads * d // 2 + 255) // 256)
    p.call("rope", [k], [m, kv, d, d, past, theta], (m * width // 2 + 255) // 256)
    stores, scales = [], []
    for side, new in (("keys", k), ("values", v)):
        store, factors = _cache(g, cache, n, width)
        stores.append(p.wrap(store))
        row = int(width * BYTES_KV[cache])
        if cache == "f32":
            codes = new
        elif cache == "f16":
            codes = p.empty(m, width, dtype=torch.float16)[1]
            p.call("cast_f32_f16", [new, codes], [m * width], (m * width // 2 + 255) // 256)
        else:
            codes, sc = p.empty(m, row, dtype=torch.uint8)[1], p.empty(m)[1]
            p.call({"q8": "quantize_q8", "q4": "quantize_q4", "fp8": "quantize_fp8_pack"}[cache], [new, codes, sc], [m, width], m)
            scales.append(p.wrap(factors))
            p.copy(scales[-1], past * 4, sc, m * 4)
            p.out[side + "_scales"] = factors[past:]
        p.copy(stores[-1], past * row, codes, m * row)
        p.out[side] = store[past:]
    dk, dv = stores
    attended, att = p.empty(m, heads * d)
    p.out["attended"] = attended
    span = min(n, window) if window else n
    if m <= 16 and span >= 512:   # few rows against many keys: the keys of a row are shared out
        split = min(64, span // 128)
        parts = [p.empty(m * heads * split, d)[1], p.empty(m * heads * split)[1], p.empty(m * heads * split)[1]]
        if cache in ("f32", "f16"):
            gqa = m == 1 and heads // kv <= 6
            p.call("attention_split_gqa" if gqa else "attention_split", [q, dk, dv, *parts],
                   [m, n, heads, kv, d, past, window, int(cache == "f16"), 1, split], m * heads * split)
        else:
            p.call(f"attention_{cache}_split", [q, dk, dv, *scales, *parts],
                   [m, n, heads, kv, d, past, window, ("q8", "q4", "fp8").index(cache), split], m * heads * split)
        p.call("attention_combine", [*parts, att], [m, heads, d, split], m * heads)
    elif cache in ("f32", "f16"):
        p.call("attention", [q, dk, dv, att], [m, n, heads, kv, d, past, 0, window, int(cache == "f16"), 1], m * heads)
    else:
        p.call(f"attention_{cache}", [q, dk, dv, *scales, att],
               [m, n, heads, kv, d, past, 0, window, ("q8", "q4", "fp8").index(cache)], m * heads)
    y, (out, dout) = p.project(c["weights"], att, wo, m, h, heads * d), p.empty(m, h)
    p.call("add", [x, y, dout], [m * h], (m * h + 255) // 256)
    p.out["hidden"] = out
    return dout


def _moe(p, g, c, x):
    m, h, f, experts, top = (c[n] for n in ("rows", "hidden", "inter", "experts", "top_k"))
    gate, up = p.weights(g, "q4k", experts * f, h), p.weights(g, "q4k", experts * f, h)
    down = p.weights(g, "q4k", experts * h, f)
    stride = f * h // 256 * 144
    logits = torch.randn(m, experts, device="cuda", generator=g)
    ids, dids = p.empty(m, top, dtype=torch.int32)
    vals, dvals = p.empty(m, top)
    phi, (out, dout) = p.empty(m * top, f)[1], p.empty(m, h)
    xn = _norm(p, g, x, m, h)
    p.call("top_k_rows", [p.wrap(logits), dids, dvals], [m, experts, top, 0], m)
    p.out.update(ids=ids, hidden=out)
    if m == 1:
        wts, sig, gate_w = p.empty(top)[1], p.empty(1)[1], p.wrap(torch.randn(h, device="cuda", generator=g) / h ** 0.5)
        p.call("moe_gate", [dvals, xn, gate_w, wts, sig], [top, h])
        p.call("moe_experts_gate_up_q4k", [xn, gate[0], up[0], dids, phi], [h, f, top, stride, stride], (f * top + 7) // 8)
        routed, shared, sphi = p.empty(h)[1], p.empty(h)[1], p.empty(f)[1]
        p.call("moe_experts_down_q4k", [phi, down[0], dids, wts, routed], [h, f, top, stride, 0], (h + 7) // 8)
        sg, su, sd = p.weights(g, "q4k", f, h), p.weights(g, "q4k", f, h), p.weights(g, "q4k", h, f)
        p.call("ffn_gate_up_silu_q4k", [xn, sg[0], su[0], sphi], [1, f, h], (f + 7) // 8)
        p.project("q4k", sphi, sd, 1, h, f, shared)
        p.call("moe_scale_add", [routed, shared, sig, dout], [h, 0], (h + 255) // 256)
    else:
        # a chunk's routing weights come from the host's router, as the candidates' softmax does there
        wts = p.wrap(torch.softmax(torch.topk(logits, top, dim=1).values, dim=1))
        p.call("moe_experts_gate_up_q4k_rows", [xn, gate[0], up[0], dids, phi], [h, f, top, stride, stride, m], (f * top + 7) // 8)
        p.call("moe_experts_down_q4k_rows", [phi, down[0], dids, wts, dout], [h, f, top, stride, 0, m], (h + 7) // 8)


def prepare(case, seed):
    p, g, c = _Program(), _gen(seed), case
    m, kind = c["rows"], c["kind"]
    if kind == "proj":
        out, dout = p.empty(m, c["n"])
        x = p.wrap(torch.randn(m, c["k"], device="cuda", generator=g))
        p.project(c["weights"], x, p.weights(g, c["weights"], c["n"], c["k"]), m, c["n"], c["k"], dout)
        p.out["y"] = out
        return p
    x = p.wrap(torch.randn(m, c["hidden"], device="cuda", generator=g))
    if kind == "head":
        logits, dlogits = p.empty(m, c["vocab"])
        ids, dids = p.empty(m, c["top_k"], dtype=torch.int32)
        vals, dvals = p.empty(m, c["top_k"])
        xn = _norm(p, g, x, m, c["hidden"])
        p.project(c["weights"], xn, p.weights(g, c["weights"], c["vocab"], c["hidden"]), m, c["vocab"], c["hidden"], dlogits)
        p.call("top_k_rows", [dlogits, dids, dvals], [m, c["vocab"], c["top_k"], 0], m)
        p.out.update(logits=logits, ids=ids, values=vals)
    elif kind == "moe":
        _moe(p, g, c, x)
    elif kind == "ffn":
        _ffn(p, g, c, x)
    elif kind == "attn":
        _attn(p, g, c, x)
    else:
        _ffn(p, g, c, _attn(p, g, c, x))
    return p


def run(state):
    for call, args in state.steps:
        call(*args)
    return state.out


# ---- what a pass cannot do without ---------------------------------------------------------------

def _proj_work(kind, m, n, k):
    return n * k // 256 * BYTES_256[kind] + (4 * n if kind == "fp8" else 0), 2 * m * n * k


def _add(*works):
    return sum(w[0] for w in works), sum(w[1] for w in works)


def _ffn_work(c):
    m, h, f = c["rows"], c["hidden"], c["inter"]
    kind = _ffn_kind(c)
    return _add(_proj_work(kind, m, f, h), _proj_work(kind, m, f, h), _proj_work(c["down"], m, h, f), (8 * m * h, 0))


def _attn_work(c):
    m, h, heads, kv, d, past, window = (c[n] for n in ("rows", "hidden", "heads", "kv_heads", "head_dim", "context", "window"))
    seen = [min(past + i + 1, window) if window else past + i + 1 for i in range(m)]
    keys = min(past + m, window + m - 1) if window else past + m
    scales = 8 if c["cache"] in ("q8", "q4", "fp8") else 0
    cache = int(keys * (2 * kv * d * BYTES_KV[c["cache"]] + scales))
    return _add(_proj_work(c["weights"], m, heads * d, h), _proj_work(c["weights"], m, kv * d, h), _proj_work(c["v"], m, kv * d, h),
                _proj_work(c["weights"], m, h, heads * d), (8 * m * h + cache, 4 * sum(seen) * heads * d))


def work(case):
    c = case
    m, kind = c["rows"], c["kind"]
    if kind == "proj":
        b, f = _add(_proj_work(c["weights"], m, c["n"], c["k"]), (4 * m * (c["n"] + c["k"]), 0))
    elif kind == "head":
        b, f = _add(_proj_work(c["weights"], m, c["vocab"], c["hidden"]), (4 * m * (c["vocab"] + c["hidden"]), 0))
    elif kind == "moe":
        used = c["experts"] * (1 - (1 - c["top_k"] / c["experts"]) ** m)   # experts that some row takes, on average
        one = 3 * _proj_work("q4k", 1, c["inter"], c["hidden"])[0]
        pairs = m * c["top_k"] + (1 if m == 1 else 0)
        b, f = int(one * (used + (1 if m == 1 else 0))) + 8 * m * c["hidden"], 6 * pairs * c["inter"] * c["hidden"]
    elif kind == "ffn":
        b, f = _ffn_work(c)
    elif kind == "attn":
        b, f = _attn_work(c)
    else:
        b, f = _add(_attn_work(c), _ffn_work(c))
    return {"bytes": b, "flops": f}


def _rounding(kind, m):
    """(2-norm, largest) relative error that the format's path shows against float64, times about four."""
    if kind == "mxfp4" and m <= 16:
        return 1e-3, 1e-2          # E4M3 activations: 2.7e-4, a code next to a tie may fall on either side
    if kind in ("mxfp4", "fp8") and m > 1:
        return 1e-4, 1e-3          # activations as sums of E4M3 terms: 2e-5
    if (kind == "q4k" and m >= 64) or (kind in ("q5k", "q6k") and m >= 17):
        return 2.4e-3, 2e-2        # operands rounded to fp16: 3e-4 a product, 6e-4 over a half layer
    return 1e-5, 2e-4              # fp32 sums: 1e-6


def tolerance(case):
    """Measured against the same launches carried out in float64, times about four."""
    c, m, kind = case, case["rows"], case["kind"]
    if kind in ("proj", "head"):
        formats = [c["weights"]]
    elif kind == "moe":            # from 17 tokens the experts' activations are rounded to fp16: 3.6e-4
        return {"rel": 1.5e-3 if m > 16 else 1e-5, "max": 1e-2 if m > 16 else 2e-4}
    else:
        formats = [c["weights"], c.get("v", c["weights"]), c.get("down", c["weights"])]
        formats.append(_ffn_kind(c) if kind == "layer" else c["weights"])
    rel, most = (max(_rounding(f, m)[i] for f in formats) for i in (0, 1))
    if kind in ("attn", "layer"):  # new cache rows: an fp16 number or a code next to a tie may fall on either side
        tile = rel > 1e-3          # the rows themselves carry fp16 rounding: 1 % of int8 codes move, 0.1 % of 4-bit ones
        if c["cache"] == "f16":
            rel, most = max(rel, 1e-4), 6e-2 if tile else 1e-2
        elif c["cache"] != "f32":
            rel, most = 8e-3 if tile else 1e-3, 0.2 if tile else 5e-2
        return {"rel": rel, "max": most, "differ": 0.01}
    return {"rel": rel, "max": most, "differ": 0.001} if kind == "head" else {"rel": rel, "max": most}
