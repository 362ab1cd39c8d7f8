"""wir::longest_first, the program order of causal attention, compiled for the
host from the device header."""
from __future__ import annotations

import os
import re
import subprocess

import pytest

from warpir_amd import kernels
from warpir_amd.lowering.cdna4 import HEADER_PATH

MAIN = r"""
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#define __device__
#define __forceinline__ inline
using std::max;
using std::min;
%s
%s
int main(int, char** v) {
  const int nx = atoi(v[1]), heads = atoi(v[2]), rev = atoi(v[3]);
  for (int hw = 0; hw < nx * heads; ++hw) {
    int x, head;
    if (rev) longest_first<true, 2048>(hw, nx, heads, x, head);
    else longest_first<false, 2048>(hw, nx, heads, x, head);
    printf("%%d %%d\n", x, head);
  }
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    with open(HEADER_PATH) as f:
        text = f.read()
    remap = re.search(r"__device__ __forceinline__ int remap_xcd.*?\n}\n", text, re.S).group(0)
    order = re.search(r"template <bool REVERSE, int TAIL>\n.*?\n}\n", text, re.S).group(0)
    d = tmp_path_factory.mktemp("order")
    src, exe = os.path.join(d, "order.cpp"), os.path.join(d, "order")
    with open(src, "w") as f:
        f.write(MAIN % (remap, order))
    subprocess.run(["g++", "-O1", "-o", exe, src], check=True)
    return exe


@pytest.mark.parametrize("reverse", [0, 1])
@pytest.mark.parametrize("nx,heads", [(1, 1), (1, 300), (3, 5), (16, 128), (16, 129), (16, 144), (32, 256), (33, 32),
                                      (64, 40), (64, 7), (300, 17), (2049, 9)])
def test_every_block_runs_once_and_the_last_heads_end_on_their_shortest_blocks(program, nx, heads, reverse):
    out = subprocess.run([program, str(nx), str(heads), str(reverse)], check=True, capture_output=True, text=True)
    order = [tuple(map(int, ln.split())) for ln in out.stdout.splitlines()]
    assert sorted(order) == [(x, h) for x in range(nx) for h in range(heads)]
    tail = min(heads, max(8, 2048 // nx // 8 * 8))
    last = order[(heads - tail) * nx:]
    assert {h for _, h in last} == set(range(heads - tail, heads))
    lengths = [x if reverse else nx - 1 - x for x, _ in last]
    assert lengths == sorted(lengths, reverse=True)
    if tail % 8 == 0 and (heads - tail) * nx % 8 == 0:   # consecutive heads on one XCD
        per = tail // 8
        for i, (_, h) in enumerate(last):
            assert (h - (heads - tail)) // per == i % 8


def test_only_causal_attention_takes_the_order():
    for name, arg in (("mha_d128_causal", "true"), ("mha_bwd_dq_d64_causal", "true"),
                      ("mha_bwd_dkdv_d128_causal_gqa", "false"), ("mha_d128", None), ("mha_bwd_dkdv_d64", None),
                      ("gemm_256_k64", None)):
        src = kernels.lowerer(name).lower(kernels.kernel(name))
        calls = re.findall(r"wir::longest_first<(\w+), 2048>", src[src.rindex('extern "C"'):])
        assert calls == ([arg] if arg else [])
