"""Piece boundaries of a decode plan (csrc/mkv_plan.h, compiled with g++) equal
a block-by-block greedy fill under the same weights. CPU only."""
from __future__ import annotations

import os
import random
import subprocess

import pytest

from mitten_amd import _build

DRIVER = r"""
#include <cstdio>
#include "mkv_plan.h"
int main() {
  int B, odd; long long cap, first;
  while (std::scanf("%d %lld %lld %d", &B, &cap, &first, &odd) == 4) {
    std::vector<int32_t> blk0(B + 1, 0), f0s;
    for (int b = 0; b < B; b++) { int n; if (std::scanf("%d", &n) != 1) return 1; blk0[b + 1] = blk0[b] + n; }
    mkv::cut_pieces(blk0.data(), B, cap, first, odd != 0, f0s);
    for (int32_t f : f0s) std::printf("%d ", f);
    std::printf("\n");
  }
}
"""


def _greedy(blocks, cap, first, odd):
    """One block at a time: 8 a block, 12 more for a sequence start inside a
    piece, at most 64 blocks; 116% of the cap for the first pieces, 96% of
    theirs for odd ones."""
    f0s, w, cnt, f = [], 0, 0, 0
    for n in blocks:
        for j in range(n):
            wi = 8 + (12 if j == 0 and cnt > 0 else 0)
            idx = len(f0s) - 1
            cq = cap * 116 // 100 if idx < first else cap
            if odd and idx & 1:
                cq = cq * 96 // 100
            if cnt > 0 and (cnt == 64 or w + wi > cq):
                cnt, w, wi = 0, 0, 8
            if cnt == 0:
                f0s.append(f)
            w += wi
            cnt += 1
            f += 1
    return f0s + [f]


@pytest.mark.parametrize("seed", range(4))
def test_cut_pieces_equals_the_block_by_block_fill(tmp_path, seed):
    src, exe = tmp_path / "cut.cpp", tmp_path / "cut"
    src.write_text(DRIVER)
    subprocess.run([os.environ.get("CXX", "g++"), "-O1", "-std=c++17", f"-I{_build.CSRC}", str(src), "-o", str(exe)],
                   check=True)
    rng = random.Random(seed)
    cases = []
    for _ in range(120):
        most = rng.choice([1, 2, 5, 70, 300])
        blocks = [rng.randint(1, most) for _ in range(rng.randint(1, 40))]
        cases.append((blocks, rng.choice([8, 9, 19, 20, 27, 28, 40, 100, rng.randint(8, 1280), 1280]),
                      rng.choice([0, 1, 3, 256]), rng.randint(0, 1)))
    text = "\n".join(f"{len(b)} {cap} {first} {odd} " + " ".join(map(str, b)) for b, cap, first, odd in cases)
    out = subprocess.run([str(exe)], input=text, capture_output=True, text=True, check=True).stdout.splitlines()
    assert len(out) == len(cases)
    for line, case in zip(out, cases):
        assert [int(x) for x in line.split()] == _greedy(*case), case
