"""The dispatch rules in sizes (csrc/dispatch.hpp), compiled for the CPU."""
import ctypes
import subprocess
from pathlib import Path

import pytest

SRC = Path(__file__).resolve().parents[1] / "knurlogic_amd" / "csrc"

SHIM = r"""
#include "dispatch.hpp"
extern "C" {
int run(int units, int tiles) { return kmi::sp_run(units, tiles); }
int place(int id, int units, int tiles, int* tile) {
    const kmi::SpPlace p = kmi::sp_place(id, units, tiles);
    *tile = p.tile;
    return p.unit;
}
int vqg(int cb, int dim, int64_t P, int64_t E, int64_t avg, int64_t H, int64_t I) {
    return kmi::vqg_wanted(cb, dim, P, E, avg, H, I);
}
int eg(int64_t active, int64_t rows, int64_t H, int64_t I) { return kmi::moe_eg_wanted(active, rows, H, I); }
int mx_batched(int64_t M, int64_t N, int64_t K) { return kmi::mx_batched_wanted(M, N, K); }
}
"""


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    d = tmp_path_factory.mktemp("rules")
    (d / "shim.cpp").write_text(SHIM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-shared", "-fPIC", f"-I{SRC}", "shim.cpp", "-o",
                    "shim.so"], cwd=d, check=True)
    L = ctypes.CDLL(str(d / "shim.so"))
    L.mx_batched.argtypes = [ctypes.c_int64] * 3
    L.eg.argtypes = [ctypes.c_int64] * 4
    L.vqg.argtypes = [ctypes.c_int] * 2 + [ctypes.c_int64] * 5
    return L


@pytest.mark.parametrize("units,tiles", [(1, 1), (1, 128), (2, 128), (4, 128), (6, 3), (8, 16), (9, 5), (16, 32), (51, 1),
                                         (3, 7), (44, 6), (20, 16), (12, 19), (6, 128), (13, 40), (100, 3)])
def test_prompt_attention_grid_covers_every_tile_once_and_fills_the_xcds(rules, units, tiles):
    n = 8 * rules.run(units, tiles)
    seen, load, t = set(), [0] * 8, ctypes.c_int()
    for i in range(n + 16):
        u = rules.place(i, units, tiles, ctypes.byref(t))
        if u < 0:
            continue
        assert 0 <= u < units and 0 <= t.value < tiles and (u, t.value) not in seen and i < n
        seen.add((u, t.value))
        load[i % 8] += 1
    assert len(seen) == units * tiles
    per_cu = lambda wgs: -(-wgs // 32)
    even = -(-units * tiles // 8)
    assert per_cu(max(load)) == per_cu(even)            # no CU has more to do than an even share gives
    if per_cu(-(-units // 8) * tiles) == per_cu(even):  # whole units then
        for i in range(n):
            u = rules.place(i, units, tiles, ctypes.byref(t))
            assert u < 0 or u % 8 == i % 8


#: measured (us): the batched kernel, the GEMM -- mxfp4, M x [N, K]
MX = [(65, 64, 2048, 12.9, 14.0), (65, 64, 14336, 16.1, 20.2), (128, 256, 4096, 12.9, 16.3), (129, 256, 14336, 19.5, 21.1),
      (65, 1000, 1024, 12.9, 13.9), (65, 1000, 4096, 14.4, 16.3), (128, 1000, 2048, 13.0, 15.3),
      (300, 64, 14336, 16.8, 20.6), (1000, 64, 14336, 19.9, 22.0),
      (65, 64, 512, 13.0, 11.0), (65, 4096, 2048, 20.2, 14.8), (1000, 256, 2048, 16.5, 15.6), (65, 1000, 14336, 27.0, 24.3),
      (300, 1000, 2048, 20.3, 17.7), (129, 1000, 4096, 18.4, 17.0), (1000, 4096, 14336, 459.5, 123.4),
      (1000, 256, 14336, 41.7, 29.0), (129, 1000, 1024, 12.0, 13.8), (1000, 256, 1024, 13.1, 14.1)]


@pytest.mark.parametrize("M,N,K,batched,gemm", MX)
def test_microscaled_products_take_the_kernel_that_measured_faster(rules, M, N, K, batched, gemm):
    assert bool(rules.mx_batched(M, N, K)) == (batched < gemm)


#: measured (us): 16-row expert tiles, the grouped GEMM -- (bytes per code or 0,
#: vector, experts, routed pairs, H, I); the points nearest to even and some others
VQ = [
    (1, 8, 16, 1920, 1024, 256, 85.9, 90.2),
    (1, 8, 128, 2048, 1536, 1024, 97.5, 102.8),
    (1, 8, 16, 4800, 1024, 512, 84.4, 89.4),
    (1, 8, 4, 1200, 1024, 512, 41.8, 79.4),
    (1, 8, 8, 1024, 1024, 512, 36.6, 76.6),
    (1, 8, 128, 2048, 2048, 768, 112.0, 103.2),
    (1, 8, 48, 2640, 1024, 768, 71.8, 65.9),
    (1, 8, 80, 1520, 1024, 512, 51.7, 47.1),
    (1, 8, 96, 1536, 2048, 512, 73.2, 66.7),
    (1, 8, 48, 14160, 2048, 768, 424.7, 238.8),
    (1, 8, 128, 3584, 2048, 768, 167.4, 125.0),
    (2, 8, 12, 324, 1024, 768, 45.4, 47.7),
    (2, 8, 16, 512, 1024, 512, 44.4, 46.8),
    (2, 8, 8, 264, 1024, 768, 46.9, 49.5),
    (2, 8, 6, 412, 2048, 512, 41.8, 70.7),
    (2, 8, 4, 512, 1024, 512, 45.3, 76.6),
    (2, 8, 64, 640, 1024, 768, 49.9, 47.1),
    (2, 8, 40, 360, 2048, 512, 56.6, 52.8),
    (2, 8, 128, 384, 2048, 768, 116.7, 108.2),
    (2, 8, 64, 448, 1536, 1024, 66.0, 60.5),
    (2, 8, 32, 704, 2048, 1536, 126.5, 69.2),
    (2, 8, 60, 7680, 2048, 768, 455.6, 136.1),
    (0, 4, 12, 756, 2048, 512, 89.7, 95.6),
    (0, 4, 8, 784, 1024, 768, 81.3, 87.1),
    (0, 4, 16, 512, 1024, 768, 55.8, 60.3),
    (0, 4, 4, 576, 1536, 512, 63.6, 95.1),
    (0, 4, 4, 400, 1280, 512, 45.1, 85.2),
    (0, 4, 20, 1160, 1536, 512, 94.5, 85.1),
    (0, 4, 96, 864, 1024, 768, 93.7, 83.5),
    (0, 4, 128, 1024, 1280, 512, 89.6, 78.9),
    (0, 4, 16, 464, 1536, 1024, 83.7, 72.7),
    (0, 4, 80, 4720, 2048, 768, 601.9, 154.1),
    (0, 4, 48, 672, 2048, 512, 89.7, 69.9),
    (0, 8, 4, 800, 3072, 512, 125.9, 133.8),
    (0, 8, 12, 600, 1024, 256, 44.1, 47.3),
    (0, 8, 16, 592, 1024, 256, 43.7, 47.2),
    (0, 8, 4, 432, 2048, 512, 55.6, 101.1),
    (0, 8, 4, 400, 1280, 512, 41.6, 81.4),
    (0, 8, 32, 768, 1280, 512, 53.8, 50.6),
    (0, 8, 32, 384, 2048, 768, 68.6, 63.3),
    (0, 8, 128, 640, 1280, 512, 72.0, 63.5),
    (0, 8, 16, 2080, 1536, 512, 109.8, 96.2),
    (0, 8, 64, 7936, 1024, 512, 314.1, 107.7),
    (0, 8, 128, 1920, 1536, 1024, 220.3, 117.5),
    (0, 2, 24, 1344, 1024, 512, 67.1, 74.8),
    (0, 2, 24, 1344, 1024, 512, 67.1, 74.8),
    (0, 2, 40, 2720, 1024, 256, 80.3, 72.5),
    (0, 2, 16, 2304, 1024, 256, 80.3, 72.4),
    (0, 2, 8, 1520, 1024, 512, 85.0, 75.6),
    (0, 2, 80, 1360, 2048, 512, 169.3, 149.6),
    (0, 2, 128, 3072, 1280, 512, 180.9, 131.0),
    (0, 2, 48, 5136, 1024, 256, 130.3, 74.3),
    (0, 2, 48, 1056, 3072, 512, 161.3, 185.2),
    (0, 8, 32, 736, 3072, 512, 117.2, 80.0),
    (0, 8, 24, 480, 2048, 768, 82.2, 62.8),
]


@pytest.mark.parametrize("cb,dim,E,P,H,I,tiles,gemm", VQ)
def test_codebook_experts_take_the_kernel_that_measured_faster(rules, cb, dim, E, P, H, I, tiles, gemm):
    avg = -(-P // min(E, P))
    assert bool(rules.vqg(cb, dim, P, E, avg, H, I)) == (gemm < tiles)


#: measured (us): moe_gemm, moe_eg -- (experts, rows each, H, I); the points nearest
#: to even and some others
EG = [
    (16, 160, 2048, 2048, 143.3, 150.5),
    (16, 170, 2048, 2048, 146.2, 157.9),
    (16, 64, 2048, 2048, 101.9, 110.0),
    (16, 80, 2048, 2048, 102.8, 111.6),
    (16, 200, 2048, 2048, 152.3, 165.5),
    (32, 96, 2048, 1024, 97.1, 106.8),
    (32, 80, 2048, 1024, 94.4, 104.4),
    (32, 200, 1536, 512, 88.4, 101.7),
    (16, 96, 2048, 2048, 105.9, 123.9),
    (32, 170, 1536, 512, 84.7, 99.2),
    (32, 180, 2048, 512, 98.7, 118.1),
    (32, 166, 1024, 512, 65.7, 88.1),
    (64, 167, 1536, 512, 144.2, 132.8),
    (40, 179, 2048, 512, 149.0, 137.1),
    (8, 591, 1536, 1024, 126.5, 114.7),
    (64, 74, 1536, 512, 89.2, 80.8),
    (64, 194, 1536, 1024, 252.2, 227.8),
    (40, 228, 2048, 1536, 323.3, 290.2),
    (128, 200, 2048, 768, 500.8, 448.8),
    (60, 160, 1920, 704, 226.5, 202.5),
    (32, 330, 2048, 1024, 299.6, 255.0),
    (32, 287, 1536, 1024, 220.5, 156.0),
    (20, 396, 1024, 768, 114.4, 99.1),
    (40, 514, 1024, 768, 260.6, 209.6),
    (24, 466, 2048, 1536, 351.3, 299.7),
]


@pytest.mark.parametrize("E,rows,H,I,gemm,eg", EG)
def test_4bit_experts_take_the_tiles_that_measured_faster(rules, E, rows, H, I, gemm, eg):
    assert bool(rules.eg(E, rows, H, I)) == (eg < gemm)
