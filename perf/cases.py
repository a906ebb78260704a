"""Timed cases of the quantized-weight path, through its public entry points.

Each case is one layer or one attention call as a model makes it:

- ``linear``: ``nn.QuantizedLinear`` over affine 4/8-bit or mxfp4/mxfp8
  weights, from one decode token to a prompt chunk;
- ``moe``: ``nn.SparseMoeBlock.experts``, the routed part of an expert block
  from the router's logits (route, gate/up, SwiGLU, down, weighted combine);
- ``vq`` / ``vq_packed``: ``nn.VQSwitchGLU.experts``, the same over
  codebook experts (byte or 16-bit codes into the layer's codebook, one scale
  per channel; bit fields with group scales and a codebook per projection,
  the artifacts' on-disk layout);
- ``decode_attention``: ``kvattn.decode_sdpa``, a decode step over the 8-bit
  KV cache's slabs;
- ``prefill_attention``: ``kvattn.quantized_sdpa``, a prompt chunk over the
  quantized cache, which longer queries than the decode kernel takes reach.

Sizes are the repository's own: the benchmark's dense shapes and 128-expert
block, the Gemma-4 artifact shape, and the prompt chunks of 512 and 2048.
"""
from __future__ import annotations

import math

import torch

from knurlogic_amd import kvattn, nn

DEV = "cuda"


def listed():
    moe = {"E": 128, "k": 8, "H": 2048, "I": 768}
    return [
        # the smallest call: one token through a square 4-bit projection
        {"name": "linear-4b-m1", "kind": "linear", "mode": "affine", "bits": 4, "group": 64,
         "M": 1, "N": 4096, "K": 4096},
        # 16 sequences decoded together through an 8-bit up projection
        {"name": "linear-8b-m16", "kind": "linear", "mode": "affine", "bits": 8, "group": 64,
         "M": 16, "N": 14336, "K": 4096},
        # a prompt chunk through a 4-bit up projection
        {"name": "linear-4b-m512", "kind": "linear", "mode": "affine", "bits": 4, "group": 64,
         "M": 512, "N": 14336, "K": 4096},
        # a ragged prompt chunk through an mxfp4 down projection
        {"name": "linear-mxfp4-m1000", "kind": "linear", "mode": "mxfp4", "bits": 4, "group": 32,
         "M": 1000, "N": 4096, "K": 14336},
        # the 4-bit expert block: one token, 16 sequences, a prompt chunk
        {"name": "moe-4b-t1", "kind": "moe", "bits": 4, "T": 1, **moe},
        {"name": "moe-4b-t16", "kind": "moe", "bits": 4, "T": 16, **moe},
        {"name": "moe-4b-t2048", "kind": "moe", "bits": 4, "T": 2048, **moe},
        # codebook experts as the artifacts ship them, one token
        {"name": "vq-packed-t1", "kind": "vq_packed", "kc": 2048, "dim": 4, "pack": 11, "group": 64, "T": 1, **moe},
        # the same, a short prompt chunk
        {"name": "vq-packed-t512", "kind": "vq_packed", "kc": 2048, "dim": 4, "pack": 11, "group": 64, "T": 512,
         **moe},
        # 16-bit codes into a layer's codebook, a full prompt chunk
        {"name": "vq-u16-t2048", "kind": "vq", "kc": 4096, "T": 2048, **moe},
        # a decode step of 4 sequences over 32k keys each
        {"name": "decode-32k", "kind": "decode_attention", "B": 4, "H": 32, "Hk": 4, "L": 1, "N": 32768, "D": 128,
         "bits": 8},
        # a prompt chunk of one sequence over 8k keys already in the cache
        {"name": "prefill-8k", "kind": "prefill_attention", "B": 1, "H": 32, "Hk": 4, "L": 512, "N": 8192, "D": 128,
         "bits": 8},
    ]


def _log(rng, lo, hi):
    """A whole number spread evenly over the logarithm of [lo, hi]."""
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def _pick(rng):
    kind = rng.choice(["linear", "linear", "linear", "moe", "moe", "vq", "vq_packed", "decode_attention",
                       "prefill_attention"])
    if kind == "linear":
        mode, bits, group = rng.choice([("affine", 4, 64), ("affine", 4, 64), ("affine", 8, 64), ("affine", 8, 64),
                                        ("affine", 4, 32), ("affine", 8, 128), ("mxfp4", 4, 32), ("mxfp8", 8, 32)])
        # widths of whole groups; outputs of any number (odd ones among them)
        K = 128 * _log(rng, 8, 112)
        N = _log(rng, 512, min(14336, 4096 * 14336 // K))
        if rng.random() < 0.7:
            N = N // 64 * 64
        return {"kind": kind, "mode": mode, "bits": bits, "group": group, "M": _log(rng, 1, 1000), "N": N, "K": K}
    if kind in ("moe", "vq", "vq_packed"):
        # experts no larger in all than 128 of 2048 -> 768 -> 2048, widths of
        # whole groups
        E, k = rng.choice([(128, 8), (128, 8), (64, 6), (32, 4), (60, 4)])
        H = 128 * rng.randint(10, 16)
        I = 64 * rng.randint(8, 12)
        T = _log(rng, 1, 512 if kind == "vq_packed" else 2048)
        c = {"kind": kind, "T": T, "E": E, "k": k, "H": H, "I": I}
        if kind == "moe":
            # 8-bit experts of 512 or 768 (a few tokens' down projection takes no other widths here)
            bits = rng.choice([4, 4, 8])
            return {**c, "bits": bits, "I": I if bits == 4 else rng.choice([512, 512 if k == 6 else 768])}
        if kind == "vq":
            # the widths that one scale per channel takes
            return {**c, "H": rng.choice([1024, 1536, 2048]), "I": rng.choice([512, 768]),
                    "kc": rng.choice([256, 4096])}
        if rng.random() < 0.3:                             # the Gemma-4 artifact's experts
            return {**c, "kc": 2048, "dim": 2, "pack": 11, "group": 64, "T": min(T, 128), "E": 128, "k": 8,
                    "H": 2816, "I": 704}
        return {**c, "kc": 2048, "dim": 4, "pack": 11, "group": 64, "I": 128 * (I // 128)}
    if kind == "decode_attention":
        B, H, Hk, D = rng.choice([(4, 32, 4, 128), (1, 32, 8, 128), (2, 16, 2, 256), (1, 64, 8, 128), (4, 16, 4, 256)])
        return {"kind": kind, "B": B, "H": H, "Hk": Hk, "L": rng.choice([1, 1, 1, 2, 4]),
                "N": _log(rng, 200, 32768 // (D // 128)), "D": D, "bits": 8}
    H, Hk, D = rng.choice([(32, 4, 128), (16, 8, 128), (16, 2, 256), (32, 8, 64)])
    L = _log(rng, 80, 512)
    return {"kind": kind, "B": 1, "H": H, "Hk": Hk, "L": L, "N": _log(rng, L, 8192 * 128 // max(D, 128)), "D": D,
            "bits": rng.choice([8, 8, 8, 4])}


def draw(rng):
    known = [{k: v for k, v in c.items() if k != "name"} for c in listed()]
    while True:
        c = _pick(rng)
        if c not in known:
            return c


# ---- inputs ------------------------------------------------------------------
# Codes and scales as quantized normal weights give them, made unpacked (what
# exact() reads) and packed to the layouts a checkpoint holds (what run() takes).

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _randn(g, *shape):
    return torch.randn(*shape, device=DEV, generator=g)


def _affine(g, shape, bits, group, std):
    """Integer codes, bf16 scales and biases of ~N(0, std) weights [..., K]."""
    top = (1 << bits) - 1
    step = top / 5.5                                       # a group spans about 5.5 deviations
    q = _randn(g, *shape).mul_(step).add_(top / 2).round_().clamp_(0, top).to(torch.uint8)
    lead = (*shape[:-1], shape[-1] // group)
    s = torch.rand(*lead, device=DEV, generator=g).mul_(0.4).add_(0.8).mul_(std / step).to(torch.bfloat16)
    b = (s.float() * (-top / 2)).to(torch.bfloat16)
    return q, s, b


def _pack_bytes(q, bits):
    """uint8 codes [..., K] -> uint32 words [..., K * bits / 32], element 0 lowest."""
    if bits == 4:
        q = q[..., 0::2] | (q[..., 1::2] << 4)
    return q.contiguous().view(torch.int32).view(torch.uint32)


def _pack_fields(c, pack):
    """int codes [..., F] -> uint32 [..., ceil(F / 32) * pack] little-endian bit fields."""
    F = c.shape[-1]
    blocks = -(-F // 32)
    if blocks * 32 != F:
        c = torch.nn.functional.pad(c, (0, blocks * 32 - F))
    c = c.view(*c.shape[:-1], blocks, 32).to(torch.int64)
    w = torch.zeros(*c.shape[:-1], pack, dtype=torch.int64, device=c.device)
    for f in range(32):
        i, sh = divmod(f * pack, 32)
        w[..., i] |= (c[..., f] << sh) & 0xFFFFFFFF
        if sh + pack > 32:
            w[..., i + 1] |= c[..., f] >> (32 - sh)
    w = torch.where(w >= 1 << 31, w - (1 << 32), w).to(torch.int32)
    return w.view(*w.shape[:-2], blocks * pack).view(torch.uint32)


_E2M1 = (0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0)


def _mx(g, N, K, bits):
    """Element codes [N, K] and E8M0 scale bytes [N, K / 32] of ~N(0, 0.02) weights."""
    w = _randn(g, N, K)
    if bits == 4:
        edges = torch.tensor([0.25, 0.75, 1.25, 1.75, 2.5, 3.5, 5.0], device=DEV)
        q = torch.bucketize(w.abs() * 2, edges).to(torch.uint8) | ((w < 0).to(torch.uint8) << 3)
    else:
        q = (w * 64).clamp_(-448, 448).to(torch.float8_e4m3fn).view(torch.uint8)
    e = torch.randint(-1, 2, (N, K // 32), device=DEV, generator=g) + (127 - 7 if bits == 4 else 127 - 12)
    return q, e.to(torch.uint8)


def _raw(case, seed):
    """Every input of a case, codes unpacked, from the seed alone."""
    g, c = _gen(seed), case
    kind = c["kind"]
    if kind == "linear":
        x = _randn(g, c["M"], c["K"]).to(torch.bfloat16)
        if c["mode"] == "affine":
            return {"x": x, "w": _affine(g, (c["N"], c["K"]), c["bits"], c["group"], 0.02)}
        return {"x": x, "w": _mx(g, c["N"], c["K"], c["bits"])}
    if kind in ("moe", "vq", "vq_packed"):
        E, H, I = c["E"], c["H"], c["I"]
        r = {"x": _randn(g, c["T"], H).to(torch.bfloat16),
             "logits": (_randn(g, c["T"], E) * 1.5).to(torch.bfloat16)}
        for name, (n, kk) in (("gate", (I, H)), ("up", (I, H)), ("down", (H, I))):
            if kind == "moe":
                r[name] = _affine(g, (E, n, kk), c["bits"], 64, 0.02)
                continue
            dim = c.get("dim", 8)
            codes = torch.randint(0, c["kc"], (E, n, kk // dim), device=DEV, generator=g, dtype=torch.int32)
            if kind == "vq_packed" or name == "gate":      # a codebook per projection, or one per layer
                book = _randn(g, c["kc"], dim).to(torch.float16)
            sshape = (E, n, kk // c["group"]) if kind == "vq_packed" else (E, n)
            scale = torch.rand(*sshape, device=DEV, generator=g).mul_(0.4).add_(0.8).mul_(0.02).to(torch.float16)
            r[name] = (codes, book, scale)
        return r
    B, H, Hk, L, N, D = (c[n] for n in ("B", "H", "Hk", "L", "N", "D"))
    cap = -(-N // 256) * 256                               # the cache's slabs grow by 256 slots
    return {"q": _randn(g, B, H, L, D).to(torch.bfloat16),
            "k": _affine(g, (B, Hk, cap, D), c["bits"], 64, 1.0),
            "v": _affine(g, (B, Hk, cap, D), c["bits"], 64, 1.0)}


def prepare(case, seed):
    c, r = case, _raw(case, seed)
    kind = c["kind"]
    if kind == "linear":
        if c["mode"] == "affine":
            q, s, b = r["w"]
            layer = nn.QuantizedLinear(_pack_bytes(q, c["bits"]), s, b, None, c["group"], c["bits"])
        else:
            q, e = r["w"]
            layer = nn.QuantizedLinear(_pack_bytes(q, c["bits"]), e, None, None, 32, c["bits"], c["mode"])
        return {"kind": kind, "layer": layer, "x": r["x"]}
    if kind == "moe":
        proj = [nn.QuantizedSwitchLinear(_pack_bytes(q, c["bits"]), s, b, None, 64, c["bits"])
                for q, s, b in (r["gate"], r["up"], r["down"])]
        return {"kind": kind, "block": nn.SparseMoeBlock(None, nn.SwitchGLU(*proj), c["k"]), "x": r["x"],
                "logits": r["logits"]}
    if kind == "vq":
        as_code = (lambda t: t.to(torch.uint8)) if c["kc"] <= 256 else (lambda t: t.to(torch.int16).view(torch.uint16))
        proj = [nn.VQSwitchLinear(as_code(q), book, s) for q, book, s in (r["gate"], r["up"], r["down"])]
        return {"kind": kind, "glu": nn.VQSwitchGLU(*proj), "x": r["x"], "logits": r["logits"], "k": c["k"]}
    if kind == "vq_packed":
        proj = [nn.VQSwitchLinear(_pack_fields(q, c["pack"]), book, s, c["group"], c["pack"], q.shape[-1] * c["dim"])
                for q, book, s in (r["gate"], r["up"], r["down"])]
        return {"kind": kind, "glu": nn.VQSwitchGLU(*proj), "x": r["x"], "logits": r["logits"], "k": c["k"]}
    N = c["N"]
    view = lambda t: tuple(p[:, :, :N] for p in (_pack_bytes(t[0], c["bits"]), t[1], t[2]))  # noqa: E731
    return {"kind": kind, "q": r["q"], "k": view(r["k"]), "v": view(r["v"]), "scale": c["D"] ** -0.5,
            "mask": "causal" if c["L"] > 1 else None, "bits": c["bits"]}


def run(state):
    s = state
    kind = s["kind"]
    if kind == "linear":
        return s["layer"](s["x"])
    if kind == "moe":
        return s["block"].experts(s["x"], s["logits"])
    if kind in ("vq", "vq_packed"):
        return s["glu"].experts(s["x"], s["logits"], s["k"])
    if kind == "decode_attention":
        return kvattn.decode_sdpa(s["q"], s["k"], s["v"], s["scale"], s["mask"], 64, 8)
    return kvattn.quantized_sdpa(s["q"], s["k"], s["v"], s["scale"], s["mask"], 64, s["bits"])


def work(case):
    c = case
    kind = c["kind"]
    if kind == "linear":
        M, N, K = c["M"], c["N"], c["K"]
        per_group = 4 if c["mode"] == "affine" else 1
        return {"bytes": N * K * c["bits"] / 8 + N * K / c["group"] * per_group + 2 * M * (N + K),
                "flops": 2 * M * N * K}
    if kind in ("moe", "vq", "vq_packed"):
        T, E, k, H, I = (c[n] for n in ("T", "E", "k", "H", "I"))
        routed = E * (1 - (1 - k / E) ** T)                # experts that some token is routed to
        rows = 2 * I + H                                   # weight rows of an expert
        if kind == "moe":
            expert = 3 * H * I * (c["bits"] / 8 + 4 / 64)
            books = 0
        elif kind == "vq":
            expert = 3 * H * I / 8 * (1 if c["kc"] <= 256 else 2) + 2 * rows
            books = c["kc"] * 16
        else:
            expert = 3 * H * I * (c["pack"] / c["dim"] / 8 + 2 / c["group"])
            books = 3 * c["kc"] * c["dim"] * 2
        return {"bytes": routed * expert + books + T * (4 * H + 2 * E), "flops": 6 * T * k * H * I}
    B, H, Hk, L, N, D = (c[n] for n in ("B", "H", "Hk", "L", "N", "D"))
    seen = N - (L - 1) / 2                                 # keys a row sees on average (causal)
    return {"bytes": 2 * B * Hk * N * D * (c["bits"] / 8 + 4 / 64) + 4 * B * H * L * D,
            "flops": 4 * B * H * L * seen * D}


def tolerance(case):
    # Against exact() the outputs are off by their own rounding to bf16 and
    # what the path rounds on the way (activations between the projections,
    # attention's scores and probabilities).
    return {"linear": {"rel": 0.01}, "moe": {"rel": 0.015}, "vq": {"rel": 0.015}, "vq_packed": {"rel": 0.015},
            "decode_attention": {"rel": 0.01}, "prefill_attention": {"rel": 0.02}}[case["kind"]]


# ---- the same in 64 bits ------------------------------------------------------

def _dequant(q, s, b, group):
    w = q.to(torch.float64).view(*q.shape[:-1], -1, group)
    return (w * s.double().unsqueeze(-1) + b.double().unsqueeze(-1)).view(q.shape)


def _mm(a, w):
    """a [m, K] times w [n, K] transposed."""
    return a @ w.t().contiguous()


def exact(case, seed):
    c, r = case, _raw(case, seed)
    kind = c["kind"]
    if kind == "linear":
        if c["mode"] == "affine":
            w = _dequant(*r["w"], c["group"])
        else:
            q, e = r["w"]
            if c["bits"] == 4:
                mag = torch.tensor(_E2M1, dtype=torch.float64, device=DEV)[(q & 7).long()]
                w = torch.where(q >= 8, -mag, mag)
            else:
                w = q.view(torch.float8_e4m3fn).to(torch.float64)
            w = (w.view(c["N"], -1, 32) * torch.exp2(e.double() - 127).unsqueeze(-1)).view(c["N"], c["K"])
        return _mm(r["x"].double(), w)
    if kind in ("moe", "vq", "vq_packed"):
        T, E, k, H = c["T"], c["E"], c["k"], c["H"]
        x, p = r["x"].double(), torch.softmax(r["logits"].double(), dim=-1)
        # ties go to the lower expert
        order = torch.sort(p, dim=-1, descending=True, stable=True).indices[:, :k]
        score = p.gather(1, order)
        score = score / score.sum(-1, keepdim=True)
        out = torch.zeros(T, H, dtype=torch.float64, device=DEV)

        def expert(name, e):
            if kind == "moe":
                q, s, b = r[name]
                return _dequant(q[e], s[e], b[e], 64)
            codes, book, s = r[name]
            w = book.double()[codes[e].long()].view(codes.shape[1], -1)
            if kind == "vq":
                return w * s[e].double().unsqueeze(-1)
            return (w.view(w.shape[0], -1, c["group"]) * s[e].double().unsqueeze(-1)).view(w.shape)

        for e in torch.unique(order).tolist():
            tok, slot = (order == e).nonzero(as_tuple=True)
            xe = x[tok]
            gate, up = _mm(xe, expert("gate", e)), _mm(xe, expert("up", e))
            y = _mm(gate * torch.sigmoid(gate) * up, expert("down", e))
            out.index_add_(0, tok, y * score[tok, slot].unsqueeze(-1))
        return out if kind == "moe" else (out, None, None)
    B, H, Hk, L, N, D = (c[n] for n in ("B", "H", "Hk", "L", "N", "D"))
    K, V = (_dequant(q[:, :, :N], s[:, :, :N], b[:, :, :N], 64) for q, s, b in (r["k"], r["v"]))
    q, rep = r["q"].double() * D ** -0.5, H // Hk
    hidden = torch.arange(N, device=DEV) > torch.arange(L, device=DEV).unsqueeze(-1) + (N - L)
    out = torch.empty(B, H, L, D, dtype=torch.float64, device=DEV)
    for b in range(B):
        for h in range(H):
            sc = _mm(q[b, h], K[b, h // rep])
            if L > 1:
                sc = sc.masked_fill(hidden, -math.inf)
            out[b, h] = torch.softmax(sc, dim=-1) @ V[b, h // rep].contiguous()
    return out
