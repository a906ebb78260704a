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
}
"""


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    d = tmp_path_factory.mktemp("rules")
    (d / "shim.cpp").write_text(SHIM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-shared", "-fPIC", f"-I{SRC}", "shim.cpp", "-o",
                    "shim.so"], cwd=d, check=True)
    L = ctypes.CDLL(str(d / "shim.so"))
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
