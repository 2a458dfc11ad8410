"""Every tile of the prefill GEMM (csrc/gemm_pair_choice.h), with and without a
k split and for both kinds of weights, that a GPT-2 model's prompts can reach is
run by tests/test_gpu_pair_gemm.py: the choice is compiled for the host and
asked for every shape of that file and for every row count of the GPT-2 widths."""
import ctypes as C
import os
import subprocess

import pytest

from tests.test_gpu_pair_gemm import MANY_ROWS, SHAPES

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = r'''
#include "gemm_pair_choice.h"
// tile * 2 + (a k split)
extern "C" int choice(int M, int N, int K, int planes, int may_split) {
  const rtg::PairChoice c = rtg::pair_choose(M, N, K, planes, may_split ? rtg::kSplitMaxFloats : 0);
  return c.tile * 2 + (c.ks > 1);
}
extern "C" int tiles() { return sizeof(rtg::kPairTiles) / sizeof(rtg::kPairTiles[0]); }
'''


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("pair_choice")
    (d / "c.cpp").write_text(SRC)
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-I", os.path.join(ROOT, "rusttorch_amd", "csrc"),
                    "-o", str(d / "libc.so"), str(d / "c.cpp")], check=True)
    return C.CDLL(str(d / "libc.so"))


def reached(lib, d, vocab, rows, planes):
    """(planes, tile, split) of a pass's GEMMs; the LM head never splits."""
    layer = [(3 * d, d), (d, d), (4 * d, d), (d, 4 * d)]
    got = [lib.choice(rows, n, k, planes, 1) for n, k in layer] + [lib.choice(rows, vocab, d, planes, 0)]
    return {(planes, g >> 1, g & 1) for g in got}


def test_the_gpu_tests_reach_every_tile(lib):
    tested = set()
    for d, _, vocab, batch, chunks in [*SHAPES, MANY_ROWS]:
        for storage in ("f32", "bf16"):
            for n in chunks:
                if storage == "f32" and batch * n <= 32 and d in (128, 768, 1024):
                    continue  # the multi-row forward
                tested |= reached(lib, d, vocab, batch * n, 2 if storage == "f32" else 1)
    real = set()
    for d in (768, 1024, 1280, 1600):
        for rows in [*range(1, 512, 8), *range(512, 4096, 64), *range(4096, 32769, 512)]:
            for planes in (1, 2):
                real |= reached(lib, d, 50257, rows, planes)
    assert len(real) == 4 * lib.tiles()  # each tile and split occurs
    assert real <= tested, sorted(real - tested)
    # the layers' epilogues (gelu to pairs, K/V, residual) on the largest tiles too
    d, _, _, batch, (n,) = MANY_ROWS
    for planes in (1, 2):
        assert {(t, s) for _, t, s in reached(lib, d, 0, batch * n, planes)} >= {(0, 0), (1, 0)}
