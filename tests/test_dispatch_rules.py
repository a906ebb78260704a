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
    return L


@pytest.mark.parametrize("units,tiles", [(1, 1), (1, 128), (2, 128), (4, 128), (6, 3), (8, 16), (9, 5), (16, 32), (51, 1),
                                         (3, 7)])
def test_prompt_attention_grid_covers_every_tile_once_and_all_xcds_alike(rules, units, tiles):
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
    assert max(load) == -(-units * tiles // 8)          # no XCD holds more than an eighth (rounded up)
    if units % 8 == 0:                                  # whole units per XCD
        for i in range(n):
            u = rules.place(i, units, tiles, ctypes.byref(t))
            assert u % 8 == i % 8


#: measured (us): the batched kernel, the GEMM -- mxfp4, M x [N, K]
MX = [(65, 64, 2048, 12.9, 14.0), (65, 64, 14336, 16.1, 20.2), (128, 256, 4096, 12.9, 16.3), (129, 256, 14336, 19.5, 21.1),
      (65, 1000, 1024, 12.9, 13.9), (65, 1000, 4096, 14.4, 16.3), (128, 1000, 2048, 13.0, 15.3),
      (300, 64, 14336, 16.8, 20.6), (1000, 64, 14336, 19.9, 22.0),
      (65, 64, 512, 13.0, 11.0), (65, 4096, 2048, 20.2, 14.8), (1000, 256, 2048, 16.5, 15.6), (65, 1000, 14336, 27.0, 24.3),
      (300, 1000, 2048, 20.3, 17.7), (129, 1000, 4096, 18.4, 17.0), (1000, 4096, 14336, 459.5, 123.4),
      (1000, 256, 14336, 41.7, 29.0)]


@pytest.mark.parametrize("M,N,K,batched,gemm", MX)
def test_microscaled_products_take_the_kernel_that_measured_faster(rules, M, N, K, batched, gemm):
    assert bool(rules.mx_batched(M, N, K)) == (batched < gemm)
