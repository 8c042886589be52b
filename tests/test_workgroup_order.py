"""Workgroup order of prefill calls (csrc/workgroup_order.h), compiled for the CPU:
the workgroups of every order together take each (query tile and chunk, sequence,
head) exactly once.
"""
import ctypes
import os
import random
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    "inkling-fa4-relative-attention_amd", "csrc")
SRC = r"""
#include "workgroup_order.h"
#include <stddef.h>
#include <vector>
using namespace ifa4;
// 0 when the workgroups of the call take every place exactly once
extern "C" int check(int heads, int group, int batch, int ragged, int chunks, int qtiles,
                     int* form) {
  const WorkgroupOrder o = workgroup_order(heads, group, batch, ragged, chunks);
  form[0] = o.lanes;
  form[1] = o.pair_heads;
  form[2] = o.lanes && !o.pair_heads ? 1 << o.spread_log : 0;
  form[3] = o.turn;
  const int qcs = qtiles * chunks;
  std::vector<int> seen((size_t)qcs * batch * heads, 0);
  const int64_t blocks = order_blocks(o) * qcs;
  for (int64_t i = 0; i < blocks; ++i) {
    WorkgroupPlace at;
    if (!workgroup_place(o, (uint32_t)i, batch, &at)) continue;
    if (at.qc < 0 || at.qc >= qcs || at.seq < 0 || at.seq >= batch || at.head < 0 ||
        at.head >= heads)
      return 1;
    if (++seen[((size_t)at.qc * batch + at.seq) * heads + at.head] != 1) return 2;
  }
  for (int n : seen)
    if (n != 1) return 3;
  return 0;
}
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("order")
    (d / "order.cpp").write_text(SRC)
    out = str(d / "order.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", f"-I{CSRC}", "-o", out,
                    str(d / "order.cpp")], check=True)
    return ctypes.CDLL(out)


def _check(lib, heads, group, batch, ragged=1, chunks=1, qtiles=3):
    form = (ctypes.c_int * 4)()
    rc = lib.check(heads, group, batch, ragged, chunks, qtiles, form)
    assert rc == 0, (heads, group, batch, ragged, chunks, qtiles)
    return dict(zip(("lanes", "pair_heads", "xcds", "turn"), form))


def test_every_place_once(lib):
    rng = random.Random(5)
    forms = set()
    for _ in range(3000):
        group = rng.choice([1, 1, 2, 3, 4, 4, 5, 6, 7, 8, 12, 16, 20, 32])
        heads = group * rng.choice([1, 1, 2, 2, 3, 4, 5, 8, 16])
        f = _check(lib, heads, group, rng.randint(1, 40), rng.randint(0, 1),
                   rng.choice([1, 1, 1, 2, 5]), rng.randint(1, 9))
        forms.add((f["lanes"], f["pair_heads"] > 0, f["xcds"], f["turn"]))
    # linear, turned, pairs, spread over 8 / 4 / 2 / 1 XCDs
    assert forms == {(0, False, 0, 0), (0, False, 0, 1), (3, True, 0, 0), (3, False, 8, 1),
                     (3, False, 4, 1), (3, False, 2, 1), (3, False, 1, 1)}
