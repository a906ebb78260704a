"""GPU parity: a prompt chunk's attention over the quantized cache in one pass
(kmi_sdpa_prefill through kvattn.quantized_sdpa) against the oracle's mlx-lm
quantized attention: tiles of 64 keys and 128 query rows and their remainders,
key splits, causal chunks that start the cache, strided slab views, both code
widths, keys far from zero (the group biases), and what stays on the separate
products.  Bar: max rel err 1e-2, cosine 0.9999 (both sides round scores to
bf16; each rounds a probability once)."""
import numpy as np
import pytest
import torch

import oracle as O
from knurlogic_amd import _abi, kvattn
from tests.util import assert_close, bf16_normal, to_numpy, to_torch, u32_to_torch

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


def _kv(rng, B, Hk, cap, D, bits, dev, mean=0.0):
    w = O.bf16_round((rng.standard_normal((B, Hk, cap, D)) + mean).astype(np.float32))
    wq, s, b = O.quantize(w, 64, bits)
    return (wq, s, b), (u32_to_torch(wq, dev), to_torch(s, dev, BF), to_torch(b, dev, BF))


@pytest.mark.parametrize("B,H,Hk,L,N,D,bits,mask", [
    (1, 2, 1, 32, 32, 128, 8, "causal"),       # 64 rows, one half-filled tile of keys, every diagonal
    (1, 4, 2, 65, 65, 128, 8, "causal"),       # rows past a tile, heads inside a row tile
    (2, 4, 1, 40, 127, 64, 8, "causal"),
    (1, 3, 3, 64, 129, 128, 4, None),
    (1, 8, 2, 50, 700, 128, 8, "causal"),      # key splits
    (1, 4, 1, 33, 1111, 256, 8, "causal"),
    (1, 2, 2, 70, 300, 256, 4, "causal"),
    (1, 2, 1, 200, 513, 64, 4, None),
])
def test_matches_the_oracle(dev, B, H, Hk, L, N, D, bits, mask):
    rng = np.random.default_rng(L + N + D + bits)
    cap = N + 19
    K, tK = _kv(rng, B, Hk, cap, D, bits, dev, 0.5)
    V, tV = _kv(rng, B, Hk, cap, D, bits, dev, -0.3)
    view = lambda t: tuple(x[:, :, :N] for x in t)
    q = bf16_normal(rng, (B, H, L, D))
    tq = to_torch(q, dev, BF)
    got = kvattn.quantized_sdpa(tq, view(tK), view(tV), D ** -0.5, mask, 64, bits)
    assert kvattn._prefill_strides(tq, view(tK), view(tV), mask, 64, bits) is not None
    ref = O.quantized_sdpa(q, view(K), view(V), D ** -0.5, mask, 64, bits)
    assert_close(to_numpy(got), ref, what="one pass")
    assert torch.equal(got, kvattn.quantized_sdpa(tq, view(tK), view(tV), D ** -0.5, mask, 64, bits))


def test_slots_past_the_keys_are_not_read_into_the_result(dev):
    """A slab's slots past N hold whatever was there: NaN scales and biases
    in them leave the result alone."""
    rng = np.random.default_rng(3)
    K, tK = _kv(rng, 1, 2, 256, 128, 8, dev)
    V, tV = _kv(rng, 1, 2, 256, 128, 8, dev)
    q = to_torch(bf16_normal(rng, (1, 4, 64, 128)), dev, BF)
    view = lambda t: tuple(x[:, :, :100] for x in t)
    before = kvattn.quantized_sdpa(q, view(tK), view(tV), 0.088, "causal")
    for t in (tK, tV):
        t[1][:, :, 100:] = float("nan")
        t[2][:, :, 100:] = float("nan")
    assert torch.equal(before, kvattn.quantized_sdpa(q, view(tK), view(tV), 0.088, "causal"))


def test_other_calls_keep_the_separate_products(dev):
    rng = np.random.default_rng(4)
    _, tK = _kv(rng, 1, 2, 96, 128, 8, dev)
    q = to_torch(bf16_normal(rng, (1, 4, 64, 128)), dev, BF)
    few = q[:, :, :4]
    add = torch.zeros(64, 96, dtype=BF, device=dev)
    short = tuple(t[:, :, :40] for t in tK)                   # causal rows that see no key
    odd = (tK[0][:, :, :, ::1].transpose(2, 3).contiguous().transpose(2, 3), *tK[1:])
    for qq, kk, mask, group in ((few, tK, "causal", 64), (q, tK, add, 64), (q, short, "causal", 64),
                                (q, odd, None, 64), (q, tK, None, 32)):
        assert kvattn._prefill_strides(qq, kk, kk, mask, group, 8) is None
    out = kvattn.quantized_sdpa(q, tK, tK, 0.1, add)
    assert_close(to_numpy(out), to_numpy(kvattn.quantized_sdpa(q, tK, tK, 0.1, None)), what="zero mask")


def test_a_row_does_not_depend_on_its_neighbours(dev):
    """One query row made 40 times larger moves that row's maximum past 8
    again and again; every other row stays what it was, bit for bit."""
    rng = np.random.default_rng(11)
    _, tK = _kv(rng, 1, 2, 1300, 128, 8, dev)
    _, tV = _kv(rng, 1, 2, 1300, 128, 8, dev)
    q = to_torch(bf16_normal(rng, (1, 4, 70, 128)), dev, BF)
    other = q.clone()
    other[0, 1, 37] *= 40
    got, ref = (kvattn.quantized_sdpa(t, tK, tV, 128 ** -0.5, "causal") for t in (other, q))
    same = torch.ones(1, 4, 70, dtype=torch.bool, device=dev)
    same[0, 1, 37] = False
    assert torch.equal(got[same], ref[same])
    assert not torch.equal(got[~same], ref[~same])


@pytest.mark.parametrize("sign", [1.0, -1.0])
@pytest.mark.parametrize("size,N,mask", [(1e30, 100, None), (1e36, 700, "causal"), (2.4e38, 100, None),
                                         (2.4e38, 700, "causal")])
def test_scores_of_any_finite_size(dev, size, sign, N, mask):
    """Scores far past float32's exponential, up to bf16's largest numbers:
    each row's softmax is 1 at its largest score, as the separate products
    give it.  Codes of 0, so a score is the sum of the group biases times the
    query; key N - 9 wins (positive) or loses least (negative) by a sixteenth,
    rows that do not see it share their weight over all keys."""
    L, D = 64, 128
    rng = np.random.default_rng(12)
    _, tV = _kv(rng, 1, 1, N, D, 8, dev)
    kb = torch.full((1, 1, N, 2), 1.0, dtype=BF, device=dev)
    kb[0, 0, N - 9] = 1.0625 if sign > 0 else 0.9375
    tK = (torch.zeros(1, 1, N, 32, dtype=torch.int32, device=dev), torch.zeros(1, 1, N, 2, dtype=BF, device=dev), kb)
    q = torch.full((1, 1, L, D), sign * size / D, dtype=BF, device=dev)
    assert kvattn._prefill_strides(q, tK, tV, mask, 64, 8) is not None
    got = kvattn.quantized_sdpa(q, tK, tV, 1.0, mask)
    V = torch.from_numpy(O.dequantize(tV[0].view(torch.int32).cpu().numpy().view(np.uint32), to_numpy(tV[1]),
                                      to_numpy(tV[2]), 64, 8)).reshape(N, D)
    ref = torch.empty(L, D)
    for l in range(L):
        last = N if mask is None else N - L + l + 1
        ref[l] = V[N - 9] if N - 9 < last else V[:last].mean(0)
    assert_close(to_numpy(got)[0, 0], ref.numpy(), what=f"scores of {sign * size}")


@pytest.mark.parametrize("mask", [None, "causal"])
def test_an_empty_batch_keeps_the_separate_products(dev, mask):
    """One query head per KV head: an empty result, as it always was."""
    rng = np.random.default_rng(13)
    _, tK = _kv(rng, 1, 2, 96, 128, 8, dev)
    none = tuple(t[:0] for t in tK)
    q = torch.empty(0, 2, 64, 128, dtype=BF, device=dev)
    assert kvattn.quantized_sdpa(q, none, none, 0.1, mask).shape == (0, 2, 64, 128)


@pytest.mark.parametrize("B,H,Hk,L,N,D,bits,mask", [
    (1, 2, 1, 32, 500, 256, 8, "causal"),      # a tile per split
    (1, 2, 1, 40, 450, 128, 4, "causal"),
    (1, 4, 2, 32, 700, 64, 8, None),
    (1, 2, 1, 36, 8200, 128, 8, "causal"),     # tens of splits
    (1, 8, 1, 1024, 600, 64, 8, None),         # enough rows for the merge by columns
])
def test_split_keys_match_the_oracle(dev, B, H, Hk, L, N, D, bits, mask):
    """Key splits down to one tile and both merges."""
    assert _abi.load().kmi_sdpa_prefill_workspace_bytes(B, H, Hk, L, N, D) > 0
    test_matches_the_oracle(dev, B, H, Hk, L, N, D, bits, mask)


@pytest.mark.parametrize("B,H,Hk,L,N,D,bits", [
    (1, 2, 1, 600, 600, 128, 8),               # L = N: rows that see nothing of a later split, whole tiles among them
    (1, 2, 2, 300, 900, 256, 8),
    (1, 1, 1, 513, 520, 64, 4),
])
def test_key_splits_that_rows_do_not_see(dev, B, H, Hk, L, N, D, bits):
    assert _abi.load().kmi_sdpa_prefill_workspace_bytes(B, H, Hk, L, N, D) > 0
    test_matches_the_oracle(dev, B, H, Hk, L, N, D, bits, "causal")


@pytest.mark.parametrize("step", [2.5, 9.0, 40.0])
@pytest.mark.parametrize("D,N,mask", [(64, 130, None), (128, 700, "causal"), (256, 330, "causal"), (128, 16384, None)])
def test_scores_that_climb_from_tile_to_tile(dev, step, D, N, mask):
    """Scores that rise by `step` per tile of 64 keys for half of the rows and
    fall for the others: the running maximum moves every few tiles, every
    tile, and by far, what was summed before it must shrink with it (also the
    biases' part, V far from zero), and key splits meet with maxima far
    apart."""
    rng = np.random.default_rng(int(step) + D + N)
    H, L = 2, 40
    u = rng.choice([-1.0, 1.0], D)
    along = (np.arange(N) / 64 - N / 128) * step / 8               # q . u / D is 8 or -8
    k = O.bf16_round((along[:, None] * u + rng.standard_normal((N, D)) * 0.3).astype(np.float32))[None, None]
    K = O.quantize(k, 64, 8)
    tK = (u32_to_torch(K[0], dev), to_torch(K[1], dev, BF), to_torch(K[2], dev, BF))
    V, tV = _kv(rng, 1, 1, N, D, 8, dev, 2.0)
    sign = np.where(np.arange(H * L) % 2, 1.0, -1.0).reshape(1, H, L, 1)
    q = O.bf16_round((8 * sign * u + rng.standard_normal((1, H, L, D))).astype(np.float32))
    got = kvattn.quantized_sdpa(to_torch(q, dev, BF), tK, tV, 1.0 / D, mask)
    ref = O.quantized_sdpa(q, K, V, 1.0 / D, mask)
    assert_close(to_numpy(got), ref, what="climbing scores")
