"""GPU parity: the dense GEMM (qmm.hip) over affine and microscaled weights
from 65 rows up, at the edges of its row and column tiles, one k-tile, and K
splits, against the oracle (max rel err 1e-2, cosine 0.9999); and the
microscaled form against the batched kernel it replaces at these sizes,
special scales and codes included."""
import numpy as np
import pytest
import torch

import oracle as O
from knurlogic_amd import ops
from tests.util import assert_close, bf16_normal, to_numpy, to_torch, u32_to_torch

pytestmark = pytest.mark.gpu
BF = torch.bfloat16

SHAPES = [  # (M, N, K): rows around a tile, ragged columns, one k-tile, K splits
    (65, 257, 64), (127, 1, 128), (128, 256, 2048), (129, 255, 576), (257, 129, 1024), (100, 1000, 4096),
]


@pytest.mark.parametrize("bits,group", [(4, 32), (4, 64), (8, 64), (8, 128)])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_affine_rows(dev, M, N, K, bits, group):
    if K % group:
        pytest.skip("K is not a multiple of the group")
    rng = np.random.default_rng(M + N + K)
    wq, s, b = O.quantize(bf16_normal(rng, (N, K), 0.02), group, bits)
    x = bf16_normal(rng, (M, K))
    got = ops.quantized_matmul(to_torch(x, dev, BF), u32_to_torch(wq, dev), to_torch(s, dev, BF), to_torch(b, dev, BF),
                               True, group, bits)
    ref = O.quantized_matmul(x, wq, s, b, True, group, bits, "float32")
    assert_close(to_numpy(got), ref, what=f"{bits}-bit {M}x{N}x{K}")


@pytest.mark.parametrize("mode", ["mxfp4", "mxfp8"])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_microscaled_rows(dev, M, N, K, mode):
    rng = np.random.default_rng(M + N + K)
    bits = 4 if mode == "mxfp4" else 8
    codes = rng.integers(0, 256, (N, K * bits // 8), dtype=np.uint8)
    if bits == 8:
        codes[(codes & 0x7f) == 0x7f] = 0x3c                # no NaN codes among the finite rows
    scales = rng.integers(120, 127, (N, K // 32), dtype=np.uint8)
    if N > 4:
        scales[0, 0], scales[1, -1] = 0, 255                # 2^-127 and NaN
        scales[2, 0] = 254                                  # 2^127: past bf16 with any larger code
        if bits == 8:
            codes[3, 5] = 0x7f                              # a NaN code
    tw = u32_to_torch(codes.view(np.uint32), dev)
    ts = torch.from_numpy(scales).to(dev)
    x = to_torch(bf16_normal(rng, (M, K)), dev, BF)
    got = to_numpy(ops.quantized_matmul(x, tw, ts, None, True, 32, bits, mode))
    ref = to_numpy(ops.qmm_batched(x, tw, ts, None, True, 32, bits, mode=mode))
    assert np.array_equal(np.isnan(got), np.isnan(ref)) and np.array_equal(np.isinf(got), np.isinf(ref))
    ok = np.isfinite(ref) & (np.abs(ref) < 1e30)
    assert_close(got[ok], ref[ok], what=f"{mode} {M}x{N}x{K}")


@pytest.mark.parametrize("mode", ["affine", "mxfp4"])
def test_up_to_128_rows_without_scratch(dev, mode):
    """A C caller that passes no workspace where the plan would split K gets
    the same product unsplit."""
    from knurlogic_amd import _abi
    rng = np.random.default_rng(5)
    M, N, K = 100, 300, 2048
    lib = _abi.load()
    x = to_torch(bf16_normal(rng, (M, K)), dev, BF)
    y = torch.empty(M, N, dtype=BF, device=dev)
    wq, s, b = O.quantize(bf16_normal(rng, (N, K), 0.02), 64, 4)
    w = u32_to_torch(wq, dev)
    st = torch.cuda.current_stream().cuda_stream
    if mode == "affine":
        ts, tb = to_torch(s, dev, BF), to_torch(b, dev, BF)
        assert lib.kmi_qmm_workspace_bytes(M, K, N, 64, 4) > 0
        rc = lib.kmi_qmm(x.data_ptr(), M, K, N, w.data_ptr(), ts.data_ptr(), tb.data_ptr(), 0, 64, 4, y.data_ptr(),
                         None, 0, st)
        ref = ops.quantized_matmul(x, w, ts, tb, True, 64, 4)
    else:
        ts = torch.full((N, K // 32), 120, dtype=torch.uint8, device=dev)
        assert lib.kmi_qmm_mx_workspace_bytes(M, K, N, 1) > 0
        rc = lib.kmi_qmm_mx(x.data_ptr(), M, K, N, w.data_ptr(), ts.data_ptr(), 0, 1, y.data_ptr(), None, 0, st)
        ref = ops.quantized_matmul(x, w, ts, None, True, 32, 4, "mxfp4")
    assert rc == 0
    assert_close(to_numpy(y), to_numpy(ref), what="no scratch")


@pytest.mark.parametrize("which", ["x", "w"])
def test_microscaled_rows_past_64_refuse_operands_off_16_bytes(dev, which):
    """kmi_qmm_mx's C contract past 64 rows (the Python wrapper copies x)."""
    from knurlogic_amd import _abi
    lib = _abi.load()
    M, N, K = 100, 300, 2048
    x = torch.zeros(M * K + 8, dtype=BF, device=dev)
    w = torch.zeros(N * K // 8 + 8, dtype=torch.int32, device=dev)
    s = torch.full((N, K // 32), 120, dtype=torch.uint8, device=dev)
    y = torch.zeros(M, N, dtype=BF, device=dev)
    ws = torch.empty(lib.kmi_qmm_mx_workspace_bytes(M, K, N, 1), dtype=torch.uint8, device=dev)
    rc = lib.kmi_qmm_mx(x.data_ptr() + (4 if which == "x" else 0), M, K, N, w.data_ptr() + (4 if which == "w" else 0),
                        s.data_ptr(), 0, 1, y.data_ptr(), ws.data_ptr(), ws.numel(), torch.cuda.current_stream().cuda_stream)
    assert rc == -1 and b"16-byte aligned" in lib.kmi_last_error()


@pytest.mark.parametrize("mode", ["mxfp4", "mxfp8"])
def test_few_microscaled_outputs_run_on_the_batched_kernel(dev, mode):
    rng = np.random.default_rng(6)
    M, N, K, bits = 100, 300, 2048, 4 if mode == "mxfp4" else 8
    w = u32_to_torch(rng.integers(0, 100, (N, K * bits // 8), dtype=np.uint8).view(np.uint32), dev)
    s = torch.from_numpy(rng.integers(115, 124, (N, K // 32), dtype=np.uint8)).to(dev)
    x = to_torch(bf16_normal(rng, (M, K)), dev, BF)
    assert torch.equal(ops.quantized_matmul(x, w, s, None, True, 32, bits, mode),
                       ops.qmm_batched(x, w, s, None, True, 32, bits, mode=mode))


@pytest.mark.parametrize("mode", ["mxfp4", "mxfp8"])
@pytest.mark.parametrize("M,N,K", [(100, 2100, 2048), (300, 700, 1024), (129, 1100, 4096)])
def test_microscaled_rows_with_k_splits(dev, M, N, K, mode):
    """Outputs enough for the GEMM, few enough that it splits K."""
    from knurlogic_amd import _abi
    assert _abi.load().kmi_qmm_mx_workspace_bytes(M, K, N, 1 if mode == "mxfp4" else 2) > 0
    test_microscaled_rows(dev, M, N, K, mode)
