"""Workgroup order of prefill calls (csrc/workgroup_order.h), compiled for the CPU:
the workgroups of every order together take each (query tile and chunk, sequence,
head) exactly once, and which calls leave the order of equal lengths.
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
extern "C" int check(int heads, int group, int batch, int ragged, int chunks, long live,
                     long slots, int windowed, int proj, int qtiles, int* form) {
  const WorkgroupOrder o = workgroup_order(OrderShape{
      heads, group, batch, ragged, qtiles, chunks, live, slots, windowed != 0, proj != 0});
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


def check_order(lib, heads, group, batch, ragged=2, chunks=1, live=1 << 20, slots=512, windowed=0,
                proj=0, qtiles=3):
    form = (ctypes.c_int * 4)()
    rc = lib.check(heads, group, batch, ragged, chunks, ctypes.c_long(live),
                   ctypes.c_long(slots), windowed, proj, qtiles, form)
    assert rc == 0, (heads, group, batch, ragged, chunks, live, windowed, proj, qtiles)
    return dict(zip(("lanes", "pair_heads", "xcds", "turn"), form))


def test_every_place_once(lib):
    rng = random.Random(5)
    forms = set()
    for _ in range(3000):
        group = rng.choice([1, 1, 2, 3, 4, 4, 5, 6, 7, 8, 12, 16, 20, 32])
        heads = group * rng.choice([1, 1, 2, 2, 3, 4, 5, 8, 16])
        f = check_order(lib, heads, group, rng.randint(1, 40), rng.randint(0, 2),
                        rng.choice([1, 1, 1, 2, 5]), rng.choice([0, 300, 511, 512, 5000]), 512,
                        rng.randint(0, 1), rng.randint(0, 1), rng.randint(1, 9))
        forms.add((f["lanes"], f["pair_heads"] > 0, f["xcds"], f["turn"]))
    # linear, turned, pairs, spread over 8 / 4 / 2 / 1 XCDs
    assert forms == {(0, False, 0, 0), (0, False, 0, 1), (3, True, 0, 0), (3, False, 8, 1),
                     (3, False, 4, 1), (3, False, 2, 1), (3, False, 1, 1)}


@pytest.mark.parametrize("heads,group,batch,kw,form", [
    # (live workgroups against resident ones, measured at workgroup_order)
    (8, 4, 16, dict(live=1101), dict(lanes=3, xcds=4, turn=1)),
    (8, 4, 6, dict(live=456), dict(lanes=0, turn=0)),          # resident at once: as equal lengths
    (8, 4, 8, dict(live=511), dict(lanes=3, pair_heads=2, turn=0)),
    (8, 4, 16, dict(live=1101, ragged=0), dict(lanes=3, pair_heads=2)),
    (8, 4, 16, dict(live=1101, chunks=3), dict(lanes=3, pair_heads=2)),
    (8, 2, 16, dict(live=1101), dict(lanes=0, turn=1)),        # groups of two: turned, not spread
    (6, 2, 12, dict(live=593), dict(lanes=0, turn=0)),         # 36 pairs: linear, as it was
    (6, 2, 16, dict(live=395), dict(lanes=3, pair_heads=3, turn=0)),
    (8, 2, 16, dict(live=1101, ragged=1), dict(lanes=3, pair_heads=4)),
    (8, 4, 16, dict(live=1101, ragged=1), dict(lanes=3, xcds=4, turn=1)),
    (8, 4, 16, dict(live=440, slots=256, proj=1), dict(lanes=3, xcds=4, turn=1)),
    (8, 2, 16, dict(live=440, slots=256, proj=1), dict(lanes=0, turn=1)),
    (8, 4, 16, dict(live=440, slots=256, proj=1, ragged=1), dict(lanes=3, pair_heads=2)),
    (8, 4, 64, dict(live=600, qtiles=1), dict(lanes=3, pair_heads=2)),
    (24, 6, 64, dict(live=5000), dict(lanes=3, pair_heads=4)),
    (8, 4, 9, dict(live=224, windowed=1), dict(lanes=3, xcds=4, turn=1)),
    (6, 3, 9, dict(live=224, windowed=1), dict(lanes=3, xcds=4, turn=1)),
    (8, 2, 9, dict(live=5000, windowed=1), dict(lanes=0, turn=0)),
    (8, 4, 9, dict(live=223, windowed=1), dict(lanes=0, turn=0)),
    (8, 4, 9, dict(live=300, windowed=1, slots=256, proj=1), dict(lanes=0, turn=0)),
    (8, 1, 6, dict(live=0, ragged=1), dict(lanes=0, turn=1)),   # eight kv heads of one head
    (4, 1, 6, dict(live=511), dict(lanes=3, pair_heads=4)),
    (16, 4, 10, dict(live=319, slots=256, proj=1), dict(lanes=3, pair_heads=4)),
    (4, 4, 12, dict(live=600), dict(lanes=3, xcds=8, turn=1)),
    (4, 4, 7, dict(live=600), dict(lanes=0, turn=0)),          # fewer sequences than XCDs
    (8, 4, 5, dict(live=5000), dict(lanes=0, turn=0)),
])
def test_order_of_a_call(lib, heads, group, batch, kw, form):
    got = check_order(lib, heads, group, batch, **kw)
    assert {k: got[k] for k in form} == form
