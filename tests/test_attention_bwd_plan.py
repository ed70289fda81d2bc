"""How the backward that keeps dS shares key blocks between workgroups (csrc/attn_bwd_plan.hpp), compiled for the host: whatever the shape
and the number of compute units, every query tile of every key block belongs to exactly one entry, and every part is written by one
and added by one."""
import ctypes
import os
import random
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SHIM = """
#include "attn_bwd_plan.hpp"
extern "C" void plan(int n_bh, int Sq, int Sk, int causal, int asked, int cus, uint32_t* items, uint32_t* merges, int* n) {
  const fo::DkdvPlan p = fo::make_dkdv_plan(n_bh, Sq, Sk, causal != 0, asked, cus);
  n[0] = p.n_items; n[1] = p.n_merges; n[2] = p.n_parts;
  for (int i = 0; i < p.n_items; ++i) items[i] = p.items[i];
  for (int i = 0; i < p.n_merges; ++i) merges[i] = p.merges[i];
}
"""


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("no host compiler")
    d = tmp_path_factory.mktemp("plan")
    (d / "shim.cpp").write_text(SHIM)
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-Wall", "-Werror", "-shared", "-fPIC", "-I", os.path.join(ROOT, "fast_ops_amd", "csrc"),
                           str(d / "shim.cpp"), "-o", str(d / "shim.so")])
    lib = ctypes.CDLL(str(d / "shim.so"))

    def call(n_bh, Sq, Sk, causal, asked=-1, cus=256):
        items, merges, n = (ctypes.c_uint32 * 96)(), (ctypes.c_uint32 * 48)(), (ctypes.c_int * 3)()
        lib.plan(n_bh, Sq, Sk, int(causal), asked, cus, items, merges, n)
        return list(items[:n[0]]), list(merges[:n[1]]), n[2]

    return call


def _check(items, merges, n_parts, Sq, Sk, causal):
    blocks, tiles = -(-Sk // 128), -(-Sq // 64)
    covered = {b: [] for b in range(blocks)}
    parts = {}
    lengths = []
    for w in items:
        blk, piece, pieces, part = w & 255, (w >> 8) & 15, (w >> 12) & 15, w >> 16
        first = min(2 * blk, tiles) if causal else 0
        n = tiles - first
        lo, hi = first + n * piece // pieces, first + n * (piece + 1) // pieces      # (as the kernel cuts them)
        covered[blk] += range(lo, hi)
        lengths.append(hi - lo)
        if pieces == 1:
            assert part == 0xFFFF and piece == 0
        else:
            assert part not in parts
            parts[part] = (blk, piece)
    for blk, got in covered.items():
        assert sorted(got) == list(range(min(2 * blk, tiles) if causal else 0, tiles))
    added = []
    for w in merges:
        blk, pieces, first = w & 255, (w >> 12) & 15, w >> 16
        added += [(first + i, (blk, i)) for i in range(pieces)]
    assert sorted(added) == sorted(parts.items()) and sorted(parts) == list(range(n_parts))
    assert all(a + 1 >= b for a, b in zip(lengths, lengths[1:]))      # longest first (a piece counts a tile more than a whole block)


def test_every_tile_once(plan):
    rng = random.Random(1)
    shared = mixed = 0
    for _ in range(4000):
        Sq, Sk = (round(2 ** rng.uniform(0, 13.2)) for _ in range(2))
        causal, asked, cus = rng.random() < 0.5, rng.choice([-1, -1, -1, 2, 3, 4]), rng.choice([256, 256, 32, 64, 304])
        items, merges, n_parts = plan(round(2 ** rng.uniform(0, 6)), Sq, Sk, causal, asked, cus)
        if not items:
            assert not merges and not n_parts
            continue
        _check(items, merges, n_parts, Sq, Sk, causal)
        shared += 1
        mixed += len({(w >> 12) & 15 for w in items}) > 1
    assert shared > 500 and mixed > 100                                # (both kinds were met: all blocks alike, and unlike ones)


def test_units_of_the_device_count(plan):
    # 128 workgroups: half of 256 units, four whole rounds of 32
    items, merges, _ = plan(4, 4096, 4096, False)
    assert merges and len(items) > 32
    assert plan(4, 4096, 4096, False, cus=32) == ([], [], 0)
    # 288 workgroups: a round and an eighth of 256 units, less than one of 304
    assert plan(12, 3072, 3072, False)[1]
    assert plan(12, 3072, 3072, False, cus=304)[0] == []
