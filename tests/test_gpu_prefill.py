"""GPU parity at prefill chunk sizes: SwitchGLU (and its weighted combine)
over the Qwen3.5-MoE expert shape -- 128 experts, top-8, 2048 -> 768 -> 2048
-- at T = 512 and 2048 tokens, for 4-bit affine experts and for VQ experts
with both codebooks (256 x 8 uint8, 4096 x 8 uint16).  The whole batch runs
on the GPU (every expert sees 32 or 128 rows); the oracle checks a sample of
tokens in full, since a token's output depends only on its own row and
experts.  Bar: max rel err 1e-2, cosine 0.9999."""
import numpy as np
import pytest
import torch

import oracle as O
from knurlogic_amd import nn
from tests.test_gpu_vq import _vq
from tests.util import assert_close, bf16_normal, to_numpy, to_torch, u32_to_torch

pytestmark = pytest.mark.gpu
BF = torch.bfloat16
E, H, I, K_TOP = 128, 2048, 768, 8


def _affine_experts(rng, bits=4):
    """4-bit g64 expert triples drawn directly in the packed layout (uniform
    codes; scales and biases of the size N(0, 0.02) weights quantize to), so
    the 600 M weights need no host-side quantization: the matmuls are what
    is checked here, the quantizer has its own bit-exact tests."""
    mats = []
    for N, Kd in ((I, H), (I, H), (H, I)):
        wq = np.frombuffer(rng.bytes(E * N * Kd * bits // 8), np.uint32).reshape(E, N, Kd * bits // 32)
        sc = O.bf16_round(rng.uniform(0.004, 0.008, (E, N, Kd // 64)).astype(np.float32))
        bi = O.bf16_round((-7.5 * sc + rng.normal(0, 0.002, sc.shape)).astype(np.float32))
        mats.append((wq, sc, bi))
    return mats


def _routing(rng, T):
    inds = np.argsort(rng.random((T, E)), axis=1)[:, :K_TOP].astype(np.int32)   # k distinct experts per token
    _, sc = O.route(bf16_normal(rng, (T, E)), K_TOP)
    return inds, sc


def _sample(rng, T, n=40):
    """Tokens checked against the oracle: the first, the last, and random ones."""
    return np.unique(np.r_[0, T - 1, rng.choice(T, n, replace=False)])


@pytest.mark.parametrize("T", [512, 2048])
def test_affine_switch_glu_at_prefill_sizes(dev, T):
    rng = np.random.default_rng(9000 + T)
    mats = _affine_experts(rng)
    q = lambda m: nn.QuantizedSwitchLinear(u32_to_torch(m[0], dev), to_torch(m[1], dev, BF),
                                           to_torch(m[2], dev, BF), None, 64, 4)
    glu = nn.SwitchGLU(*(q(m) for m in mats))
    fns = [lambda xs, e, m=m: O.quantized_matmul(xs, m[0][e], m[1][e], m[2][e], True, 64, 4, "bfloat16")
           for m in mats]
    x = bf16_normal(rng, (T, H))
    inds, sc = _routing(rng, T)
    tx, ti = to_torch(x, dev, BF), torch.from_numpy(inds).to(dev)
    got = to_numpy(glu(tx, ti))
    comb = to_numpy(glu.combine(tx, ti, to_torch(sc, dev, BF)))
    assert got.shape == (T, K_TOP, H) and np.isfinite(got).all()
    s = _sample(rng, T)
    ref = O.switch_glu(x[s], inds[s], *fns)
    assert_close(got[s], ref, what=f"affine switch_glu T={T}")
    assert_close(comb[s], O.combine(ref, sc[s]), what=f"affine combine T={T}")


@pytest.mark.parametrize("kc", [256, 4096])
@pytest.mark.parametrize("T", [512, 2048])
def test_vq_switch_glu_at_prefill_sizes(dev, T, kc):
    rng = np.random.default_rng(9100 + T + kc)
    (hg, gg), (hu, gu), (hd, gd) = [_vq(rng, E, n, kd, kc, 0, dev) for n, kd in ((I, H), (I, H), (H, I))]
    # one codebook for the layer, as the VQ artifacts ship it
    hu, hd = (hu[0], hg[1], hu[2]), (hd[0], hg[1], hd[2])
    gu, gd = (gu[0], gg[1], gu[2]), (gd[0], gg[1], gd[2])
    glu = nn.VQSwitchGLU(*(nn.VQSwitchLinear(*g) for g in (gg, gu, gd)))
    x = bf16_normal(rng, (T, H))
    inds, sc = _routing(rng, T)
    tx, ti = to_torch(x, dev, BF), torch.from_numpy(inds).to(dev)
    got = to_numpy(glu(tx, ti))
    comb = to_numpy(glu.combine(tx, ti, to_torch(sc, dev, BF)))
    assert got.shape == (T, K_TOP, H) and np.isfinite(got).all()
    s = _sample(rng, T)
    fn = lambda h: (lambda xs, e: O.vq_matmul(xs, h[0][e], h[1], h[2][e], 0, "bfloat16"))
    ref = O.switch_glu(x[s], inds[s], fn(hg), fn(hu), fn(hd))
    assert_close(got[s], ref, what=f"vq switch_glu T={T} kc={kc}")
    assert_close(comb[s], O.combine(ref, sc[s]), what=f"vq combine T={T} kc={kc}")


@pytest.mark.parametrize("bits", [4, 8])
def test_grouped_gemm_with_k_tiles_past_a_group(dev, bits):
    """The grouped expert GEMM (from 64 routed rows per expert) on experts
    whose K runs 9 (gate/up, H = 576) and 5 (down, I = 320) k-tiles, which
    end part-way through the 4-deep load ring; 8 experts, top-2, 512 tokens
    (128 rows per expert)."""
    rng = np.random.default_rng(9200 + bits)
    e, h, i_, k, T = 8, 576, 320, 2, 512
    mats = []
    for N, Kd in ((i_, h), (i_, h), (h, i_)):
        wq = np.frombuffer(rng.bytes(e * N * Kd * bits // 8), np.uint32).reshape(e, N, Kd * bits // 32)
        sc = O.bf16_round(rng.uniform(0.004, 0.008, (e, N, Kd // 64)).astype(np.float32) / (1 << (bits - 4)))
        bi = O.bf16_round((-0.5 * ((1 << bits) - 1) * sc + rng.normal(0, 0.002, sc.shape)).astype(np.float32))
        mats.append((wq, sc, bi))
    q = lambda m: nn.QuantizedSwitchLinear(u32_to_torch(m[0], dev), to_torch(m[1], dev, BF),
                                           to_torch(m[2], dev, BF), None, 64, bits)
    glu = nn.SwitchGLU(*(q(m) for m in mats))
    fns = [lambda xs, ex, m=m: O.quantized_matmul(xs, m[0][ex], m[1][ex], m[2][ex], True, 64, bits, "bfloat16")
           for m in mats]
    x = bf16_normal(rng, (T, h))
    inds = np.argsort(rng.random((T, e)), axis=1)[:, :k].astype(np.int32)
    got = to_numpy(glu(to_torch(x, dev, BF), torch.from_numpy(inds).to(dev)))
    assert got.shape == (T, k, h) and np.isfinite(got).all()
    s = _sample(rng, T)
    assert_close(got[s], O.switch_glu(x[s], inds[s], *fns), what=f"grouped gemm {bits}-bit")


@pytest.mark.parametrize("h,i_,group", [(320, 1984, 64), (256, 2048, 128), (64, 2048, 64)])
def test_expert_tiles_at_their_edges(dev, h, i_, group):
    """4-bit experts of uneven rows, 16 of them (one round of the grouped
    GEMM; over 64 experts below: the tiles whose work follows their rows,
    moe_eg.hip): row counts around moe_eg's 32-row blocks and its largest
    tile, an expert without rows, columns that do not fill a column block,
    one and several K stages, pairs whose expert is out of range."""
    rng = np.random.default_rng(9300 + h)
    counts = [1, 31, 32, 33, 64, 65, 95, 127, 128, 129, 159, 160, 161, 330, 0, 40]
    e = len(counts)
    mats = []
    for N, Kd in ((i_, h), (i_, h), (h, i_)):
        wq = np.frombuffer(rng.bytes(e * N * Kd // 2), np.uint32).reshape(e, N, Kd // 8)
        sc = O.bf16_round(rng.uniform(0.004, 0.008, (e, N, Kd // group)).astype(np.float32))
        bi = O.bf16_round((-7.5 * sc + rng.normal(0, 0.002, sc.shape)).astype(np.float32))
        mats.append((wq, sc, bi))
    q = lambda m: nn.QuantizedSwitchLinear(u32_to_torch(m[0], dev), to_torch(m[1], dev, BF),
                                           to_torch(m[2], dev, BF), None, group, 4)
    glu = nn.SwitchGLU(*(q(m) for m in mats))
    inds = np.concatenate([np.full(n, x) for x, n in enumerate(counts)] + [[e, -1]]).astype(np.int32)
    rng.shuffle(inds)
    x = bf16_normal(rng, (len(inds), h))
    tx, ti = to_torch(x, dev, BF), torch.from_numpy(inds[:, None]).to(dev)
    got = glu(tx, ti)
    assert torch.equal(got, glu(tx, ti)), "a repeated call differs"
    y, bad = to_numpy(got)[:, 0], (inds < 0) | (inds >= e)
    assert (y[bad] == 0).all()
    fns = [lambda xs, ex, m=m: O.quantized_matmul(xs, m[0][ex], m[1][ex], m[2][ex], True, group, 4, "bfloat16")
           for m in mats]
    assert_close(y[~bad], O.switch_glu(x[~bad], inds[~bad, None], *fns)[:, 0], what="expert tiles")


@pytest.mark.parametrize("what", ["none", "x", "s_gu", "b_gu", "s_down", "b_down"])
def test_expert_operands_at_any_element_offset(dev, what):
    """64 experts of about 70 rows (moe_eg's sizes): operands that are views
    off the alignment its loads need -- a scale or bias tensor at an odd
    element, x at a 4-byte offset -- give the same result."""
    from knurlogic_amd import ops
    rng = np.random.default_rng(9400)
    e, h, i_, k, T = 64, 320, 768, 4, 1120
    t = {}
    for name, N, Kd in (("gu", 2 * i_, h), ("down", h, i_)):
        wq = np.frombuffer(rng.bytes(e * N * Kd // 2), np.uint32).reshape(e, N, Kd // 8)
        sc = O.bf16_round(rng.uniform(0.004, 0.008, (e, N, Kd // 64)).astype(np.float32))
        bi = O.bf16_round((-7.5 * sc + rng.normal(0, 0.002, sc.shape)).astype(np.float32))
        t.update({f"w_{name}": u32_to_torch(wq, dev), f"s_{name}": to_torch(sc, dev, BF), f"b_{name}": to_torch(bi, dev, BF)})
        if name == "gu":
            gu = (wq, sc, bi)
        else:
            down = (wq, sc, bi)
    x = bf16_normal(rng, (T, h))
    t["x"] = to_torch(x, dev, BF)
    if what != "none":
        off = 2 if what == "x" else 1
        flat = torch.empty(t[what].numel() + off, dtype=BF, device=dev)
        view = flat[off:].view(t[what].shape)
        view.copy_(t[what])
        t[what] = view
    inds = np.argsort(rng.random((T, e)), axis=1)[:, :k].astype(np.int32)
    got = to_numpy(ops.switch_glu(t["x"], torch.from_numpy(inds).to(dev), t["w_gu"], t["s_gu"], t["b_gu"], t["w_down"],
                                  t["s_down"], t["b_down"]))
    part = lambda m, lo, hi: (lambda xs, ex: O.quantized_matmul(xs, m[0][ex, lo:hi], m[1][ex, lo:hi], m[2][ex, lo:hi],
                                                                True, 64, 4, "bfloat16"))
    s = _sample(rng, T)
    ref = O.switch_glu(x[s], inds[s], part(gu, 0, i_), part(gu, i_, 2 * i_), part(down, 0, h))
    assert_close(got[s], ref, what=f"{what} off its alignment")


@pytest.mark.parametrize("h,i_,group", [(320, 768, 64), (1024, 640, 128), (128, 704, 64)])
def test_expert_tiles_at_their_edges_over_many_experts(dev, h, i_, group):
    """As test_expert_tiles_at_their_edges over 64 experts, which the dispatch
    puts on the tiles whose work follows their rows (the library's own query;
    16 experts fit one round of the grouped GEMM)."""
    from knurlogic_amd import _abi
    rng = np.random.default_rng(9500 + h)
    counts = [1, 31, 32, 33, 64, 65, 95, 127, 128, 129, 159, 160, 161, 330, 0] + [60] * 49
    e, T = len(counts), sum(counts) + 2
    i_ = i_ // group * group
    assert _abi.load().kmi_switch_glu_tile_rows(T, h, i_, 1, e, group, 4) == 160
    mats = []
    for N, Kd in ((i_, h), (i_, h), (h, i_)):
        wq = np.frombuffer(rng.bytes(e * N * Kd // 2), np.uint32).reshape(e, N, Kd // 8)
        sc = O.bf16_round(rng.uniform(0.004, 0.008, (e, N, Kd // group)).astype(np.float32))
        bi = O.bf16_round((-7.5 * sc + rng.normal(0, 0.002, sc.shape)).astype(np.float32))
        mats.append((wq, sc, bi))
    q = lambda m: nn.QuantizedSwitchLinear(u32_to_torch(m[0], dev), to_torch(m[1], dev, BF),
                                           to_torch(m[2], dev, BF), None, group, 4)
    glu = nn.SwitchGLU(*(q(m) for m in mats))
    inds = np.concatenate([np.full(n, x) for x, n in enumerate(counts)] + [[e, -1]]).astype(np.int32)
    rng.shuffle(inds)
    x = bf16_normal(rng, (len(inds), h))
    tx, ti = to_torch(x, dev, BF), torch.from_numpy(inds[:, None]).to(dev)
    got = glu(tx, ti)
    assert torch.equal(got, glu(tx, ti)), "a repeated call differs"
    y, bad = to_numpy(got)[:, 0], (inds < 0) | (inds >= e)
    assert (y[bad] == 0).all()
    fns = [lambda xs, ex, m=m: O.quantized_matmul(xs, m[0][ex], m[1][ex], m[2][ex], True, group, 4, "bfloat16")
           for m in mats]
    assert_close(y[~bad], O.switch_glu(x[~bad], inds[~bad, None], *fns)[:, 0], what="expert tiles")


def test_experts_that_fit_one_round_stay_on_the_grouped_gemm():
    """(The library's host query; no GPU work.)"""
    from knurlogic_amd import _abi
    rows = lambda T, H, I, k, E: _abi.load().kmi_switch_glu_tile_rows(T, H, I, k, E, 64, 4)
    assert rows(768, 2048, 2048, 2, 16) == 128 and rows(1328, 1024, 512, 4, 32) == 256
    assert rows(2048, 2048, 768, 8, 128) == 160 and rows(1, 2048, 768, 8, 128) == 1
