"""How the pipelined forward kernel shares the keys of query blocks between workgroups (csrc/attn_fwd_plan.hpp), compiled for the host:
whatever the shape and the number of workgroups the device holds, every key tile of every block belongs to exactly one entry, a causal
block's last entry reaches far enough back for each of its rows to see a key, and every part is written by one and added by one."""
import ctypes
import math
import os
import random
import shutil
import subprocess
import time

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SHIM = """
#include "attn_fwd_plan.hpp"
extern "C" void plan(int n_bh, int Sq, int Sk, int causal, int asked, int slots, uint32_t* items, uint32_t* merges, int* n) {
  const fo::DkdvPlan p = fo::make_fwd_plan(n_bh, Sq, Sk, causal != 0, asked, slots);
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

    def call(n_bh, Sq, Sk, causal, asked=-1, slots=256):
        items, merges, n = (ctypes.c_uint32 * 96)(), (ctypes.c_uint32 * 48)(), (ctypes.c_int * 3)()
        lib.plan(n_bh, Sq, Sk, int(causal), asked, slots, items, merges, n)
        return list(items[:n[0]]), list(merges[:n[1]]), n[2]

    return call


def _check(items, merges, n_parts, Sq, Sk, causal):
    blocks, keys = -(-Sq // 128), -(-Sk // 64)
    covered, parts = {b: [] for b in range(blocks)}, {}
    for w in items:
        blk, piece, pieces, part = w & 255, (w >> 8) & 15, (w >> 12) & 15, w >> 16
        n = min(keys, 2 * (blk + 1)) if causal else keys
        lo, hi = n * piece // pieces, n * (piece + 1) // pieces
        assert 0 <= piece < pieces <= 4 and lo < hi
        if causal:
            assert lo * 64 <= blk * 128                         # the block's first row sees the piece's first key
        covered[blk] += range(lo, hi)
        if pieces == 1:
            assert part == 0xFFFF
        else:
            assert part < n_parts and part not in parts
            parts[part] = (blk, piece, pieces)
    for b in range(blocks):
        assert sorted(covered[b]) == list(range(min(keys, 2 * (b + 1)) if causal else keys))
    seen = []
    for m in merges:
        blk, pieces, first = m & 0xFFF, (m >> 12) & 15, m >> 16
        for i in range(pieces):
            assert parts[first + i] == (blk, i, pieces)
            seen.append(first + i)
    assert sorted(seen) == list(range(n_parts)) == sorted(parts)


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("asked", [-1, 2, 3, 4])
def test_every_key_tile_once(plan, causal, asked):
    rng = random.Random(asked + 10 * causal)
    shared = 0
    for _ in range(400):
        Sq, Sk = rng.randint(1, 6000), rng.randint(1, 9000)
        if rng.random() < 0.5:
            Sk = Sq
        items, merges, n_parts = plan(rng.choice([1, 2, 4, 6, 8, 12, 32]), Sq, Sk, causal, asked, rng.choice([256, 512, 304, 8]))
        if merges:
            shared += 1
            _check(items, merges, n_parts, Sq, Sk, causal)
    assert shared > 50


def test_where_blocks_are_shared(plan):
    assert plan(8, 3000, 3000, True)[1] and plan(6, 4096, 4096, True)[1] and plan(4, 4096, 4096, False)[1] and plan(12, 3072, 3072, False)[1]
    assert not plan(8, 3000, 3000, True, 0)[1]                  # switched off
    assert not plan(32, 8192, 8192, True)[1] and not plan(12, 256, 256, True)[1] and not plan(12, 4096, 4096, False)[1]


def test_shapes_in_turn_do_not_plan_anew():
    """A model of many lengths asks in turn: how the query blocks are shared is worked out once for each (up to 12 us), not at every call."""
    from fast_ops_amd import _lib

    ask = _lib.load().fo_attn_fwd_workspace
    strides = (ctypes.c_int64 * 3)(0, 1 << 21, 128)

    def per_call(lengths):
        best = math.inf
        for _ in range(7):
            t0 = time.perf_counter()
            for _ in range(2000 // len(lengths)):
                for n in lengths:
                    ask(1, 6, n, n, 128, strides, strides, 1)
            best = min(best, (time.perf_counter() - t0) / (2000 // len(lengths) * len(lengths)))
        return best

    one = per_call([4096] * 24)
    assert per_call([4096 - 64 * i for i in range(24)]) < 3.0 * one
