"""GPU parity: the expert-grouped codebook GEMM (vq_gemm.hip: SwitchGLU over VQ
experts at prefill sizes) against the oracle's exact decode-then-matmul, at
the edges of its 32-row blocks and largest tiles (one row, one short of a
block, one past the largest tile), with columns that do not fill a column
block, several K stages, pairs whose expert is out of range, and the layouts
of the codes.  64 experts reach it; the same edges over 6 experts, which the
dispatch leaves on the 16-row expert tiles, stand first.  Bar: max rel err 1e-2, cosine 0.9999."""
import numpy as np
import pytest
import torch

import oracle as O
from knurlogic_amd import nn
from tests.test_gpu_vq import _vq
from tests.test_gpu_vq_packed import _packed
from tests.util import assert_close, bf16_normal, to_numpy, to_torch

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


def _check(rng, dev, glu, fns, counts, H):
    """Pairs in random order over experts of the given row counts, and three
    whose expert does not exist."""
    E = len(counts)
    inds = np.concatenate([np.full(n, e) for e, n in enumerate(counts)] + [[E, -1, E + 7]]).astype(np.int32)
    rng.shuffle(inds)
    inds = inds[:, None]
    x = bf16_normal(rng, (len(inds), H))
    tx, ti = to_torch(x, dev, BF), torch.from_numpy(inds).to(dev)
    got = glu(tx, ti)
    again = glu(tx, ti)
    assert torch.equal(got, again), "a repeated call differs"
    y = to_numpy(got)[:, 0]
    bad = (inds[:, 0] < 0) | (inds[:, 0] >= E)
    assert (y[bad] == 0).all()
    ref = O.switch_glu(x[~bad], inds[~bad], *fns)[:, 0]
    assert_close(y[~bad], ref, what="vq gemm")
    scores = to_torch(rng.uniform(0.1, 1.0, inds.shape), dev, BF)
    comb = to_numpy(glu.combine(tx, ti, scores))
    assert_close(comb[~bad], O.combine(ref[:, None], to_numpy(scores)[~bad]), what="vq gemm combine")


@pytest.mark.parametrize("kc,shared,H,I", [(256, True, 512, 768), (256, False, 768, 512), (200, False, 1024, 512),
                                           (4096, True, 512, 768), (1024, False, 1024, 512)])
def test_per_channel_scales(dev, kc, shared, H, I):
    rng = np.random.default_rng(kc + H + I)
    counts = [1, 31, 33, 160, 161, 650]
    E = len(counts)
    (hg, gg), (hu, gu), (hd, gd) = [_vq(rng, E, n, kd, kc, 0, dev) for n, kd in ((I, H), (I, H), (H, I))]
    if shared:
        hu, gu = (hu[0], hg[1], hu[2]), (gu[0], gg[1], gu[2])
    glu = nn.VQSwitchGLU(*(nn.VQSwitchLinear(*g) for g in (gg, gu, gd)))
    fn = lambda h: (lambda xs, e: O.vq_matmul(xs, h[0][e], h[1], h[2][e], 0, "bfloat16"))
    _check(rng, dev, glu, (fn(hg), fn(hu), fn(hd)), counts, H)


@pytest.mark.parametrize("bits,kc,dim,group,H,I", [(11, 2048, 4, 64, 384, 256), (11, 2048, 2, 64, 192, 320),
                                                   (16, 3000, 4, 64, 256, 128), (9, 300, 8, 128, 256, 512),
                                                   (12, 4096, 4, 128, 128, 640), (8, 256, 2, 64, 64, 128)])
def test_packed_fields(dev, bits, kc, dim, group, H, I):
    rng = np.random.default_rng(bits + H + I)
    counts = [1, 31, 33, 127, 129, 800]
    E = len(counts)
    (hg, gg), (hu, gu), (hd, gd) = [_packed(rng, E, n, kd, dim, kc, bits, group, dev)
                                    for n, kd in ((I, H), (I, H), (H, I))]
    glu = nn.VQSwitchGLU(*(nn.VQSwitchLinear(*g, group, bits) for g in (gg, gu, gd)))
    fn = lambda h: (lambda xs, e: O.vq_packed_matmul(xs, h[0][e], h[1], h[2][e], bits, group, "bfloat16"))
    _check(rng, dev, glu, (fn(hg), fn(hu), fn(hd)), counts, H)


# The same over experts enough for the dispatch to take the grouped GEMM, which
# the library's own query confirms (6 experts leave most of the GPU idle and run
# on the 16-row tiles).
MANY = 64


@pytest.mark.parametrize("kc,shared,H,I", [(256, True, 1024, 512), (256, False, 768, 512), (200, False, 1024, 512),
                                           (4096, True, 512, 512), (1024, False, 1024, 512)])
def test_per_channel_scales_over_many_experts(dev, kc, shared, H, I):
    from knurlogic_amd import _abi
    rng = np.random.default_rng(kc + H + I + 1)
    counts = [1, 31, 32, 33, 159, 160, 161, 330, 0] + [20] * (MANY - 9)
    P = sum(counts) + 3
    assert _abi.load().kmi_vq_switch_glu_tile_rows(P, H, I, 1, MANY, 1 if kc <= 256 else 2, kc, shared) == 160
    (hg, gg), (hu, gu), (hd, gd) = [_vq(rng, MANY, n, kd, kc, 0, dev) for n, kd in ((I, H), (I, H), (H, I))]
    if shared:
        hu, gu = (hu[0], hg[1], hu[2]), (gu[0], gg[1], gu[2])
    glu = nn.VQSwitchGLU(*(nn.VQSwitchLinear(*g) for g in (gg, gu, gd)))
    fn = lambda h: (lambda xs, e: O.vq_matmul(xs, h[0][e], h[1], h[2][e], 0, "bfloat16"))
    _check(rng, dev, glu, (fn(hg), fn(hu), fn(hd)), counts, H)


@pytest.mark.parametrize("bits,kc,dim,group,H,I", [(11, 2048, 4, 64, 384, 256), (11, 2048, 2, 64, 192, 320),
                                                   (16, 3000, 4, 64, 256, 128), (9, 300, 8, 128, 256, 512),
                                                   (12, 4096, 4, 128, 128, 640), (8, 256, 2, 64, 64, 128)])
def test_packed_fields_over_many_experts(dev, bits, kc, dim, group, H, I):
    from knurlogic_amd import _abi
    rng = np.random.default_rng(bits + H + I + 1)
    tile = 64 if dim == 2 else 128
    counts = [1, 31, 32, 33, tile - 1, tile, tile + 1, 2 * tile + 40, 0] + [25] * (MANY - 9)
    P = sum(counts) + 3
    assert _abi.load().kmi_vq_packed_switch_glu_tile_rows(P, H, I, 1, MANY, bits, kc, dim, group, 0) == tile
    (hg, gg), (hu, gu), (hd, gd) = [_packed(rng, MANY, n, kd, dim, kc, bits, group, dev)
                                    for n, kd in ((I, H), (I, H), (H, I))]
    glu = nn.VQSwitchGLU(*(nn.VQSwitchLinear(*g, group, bits) for g in (gg, gu, gd)))
    fn = lambda h: (lambda xs, e: O.vq_packed_matmul(xs, h[0][e], h[1], h[2][e], bits, group, "bfloat16"))
    _check(rng, dev, glu, (fn(hg), fn(hu), fn(hd)), counts, H)


def test_few_experts_stay_on_the_small_tiles():
    """(The library's host query; no GPU work.)"""
    from knurlogic_amd import _abi
    L = _abi.load()
    assert L.kmi_vq_switch_glu_tile_rows(1024, 1024, 512, 2, 8, 1, 256, 1) == 16
    assert L.kmi_vq_switch_glu_tile_rows(512, 2048, 768, 2, 8, 2, 4096, 1) == 16
    assert L.kmi_vq_packed_switch_glu_tile_rows(400, 1280, 512, 2, 8, 11, 2048, 4, 64, 0) == 16
    assert L.kmi_vq_switch_glu_tile_rows(2048, 2048, 768, 8, 128, 2, 4096, 1) == 160
    assert L.kmi_vq_packed_switch_glu_tile_rows(512, 2048, 768, 8, 128, 11, 2048, 4, 64, 0) == 128
    assert L.kmi_vq_switch_glu_tile_rows(1, 2048, 768, 8, 128, 1, 256, 1) == 1
