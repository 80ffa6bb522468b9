"""The dense prefill schedule, run on the host: every (head, row block) is taken once, and a causal call whose
heads divide by the 8 XCDs loads them alike, each from its heaviest blocks to its lightest."""
import collections
import ctypes
import os
import random
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "cuda-attention-kernels_amd", "csrc")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
SOURCE = """
#include "fa_prefill_common.hpp"
extern "C" void schedule(int heads_kv, int group, int nq, int nk, int head_dim, int n_rowblk, int causal, int nw, int* out) {
  fa::TileArgs a{};
  a.kv_groups = heads_kv;
  a.group = group;
  a.nq = nq;
  a.nk = nk;
  a.causal = causal;
  a.n_rowblk = n_rowblk;
  a.total = heads_kv * group * n_rowblk;
  fa::prefill_schedule(a, head_dim, nw);
  *out++ = a.u_heads;
  *out++ = a.deal;
  for (int i = 0; i < a.total; ++i) {
    const fa::PrefillOrder o = fa::prefill_dense_order(a, (uint32_t)i);
    *out++ = (int)o.head;
    *out++ = (int)o.rank;
  }
}
"""


@pytest.fixture(scope="module")
def schedule(tmp_path_factory):
    d = tmp_path_factory.mktemp("schedule")
    src, lib = d / "schedule.hip", d / "libschedule.so"
    src.write_text(SOURCE)
    subprocess.run([HIPCC, "--offload-host-only", "-std=c++17", "-O1", "-fPIC", "-shared", "-I", CSRC, "-x", "hip", str(src),
                    "-o", str(lib)], check=True, capture_output=True)
    c = ctypes.CDLL(str(lib)).schedule

    def run(heads_kv, group, n, d, causal, nw=4, nk=None):
        n_rowblk = -(-n // (32 * nw))
        total = heads_kv * group * n_rowblk
        out = (ctypes.c_int * (2 + 2 * total))()
        c(heads_kv, group, n, nk or n, d, n_rowblk, int(causal), nw, out)
        items = list(zip(out[2::2], out[3::2]))
        assert sorted(items) == [(h, r) for h in range(heads_kv * group) for r in range(n_rowblk)]
        run.dealt = bool(out[1])
        return items, out[0], n_rowblk

    return run


SHAPES = [(1, 1, 1), (1, 8, 4), (3, 8, 4), (7, 4, 4), (6, 8, 4), (3, 1, 8), (8, 8, 4), (11, 8, 1), (10, 32, 1), (3, 8, 8), (5, 5, 4), (4, 11, 3),
          (1, 3, 3), (2, 3, 4), (13, 8, 1)]


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("d", [32, 64, 128, 256])
def test_every_block_once(schedule, d, causal):
    rng = random.Random(d)
    for b, hkv, group in SHAPES:
        for n in (1, 128, 129, rng.randrange(130, 3000), 1999):
            schedule(b * hkv, group, n, d, causal, 4)
    schedule(32, 4, 4096, 128, causal, 8)


@pytest.mark.parametrize("n", [257, 600, 700, 1024, 1400, 1999])
@pytest.mark.parametrize("b,hkv,group", [s for s in SHAPES if s[0] * s[1] * s[2] % 8 == 0])
def test_xcds_share_causal_work_evenly(schedule, b, hkv, group, n):
    items, unit, n_rowblk = schedule(b * hkv, group, n, 128, True)
    own = [items[x::8] for x in range(8)]  # workgroup i runs on XCD i % 8
    ranks = [collections.Counter(r for _, r in x) for x in own]
    assert all(r == ranks[0] for r in ranks)
    for x in own:
        x = x[31::-1] + x[32:] if 256 < len(items) <= 512 else x  # (the first 32 are taken in reverse)
        assert x[0][1] == 0 and x[-1][1] == n_rowblk - 1  # from a heaviest to a lightest block
        # within a unit the ranks go down; a unit starts over at most once every `unit` heads
        assert sum(p[1] > q[1] for p, q in zip(x, x[1:])) == -(-(b * hkv * group // 8) // unit) - 1


@pytest.mark.parametrize("heads_kv,group,nq,nk,d,dealt", [
    (28, 1, 1300, 1300, 128, True), (84, 1, 1500, 1500, 64, True), (108, 1, 1500, 1500, 128, False),
    (35, 4, 178, 565, 64, False), (35, 4, 565, 565, 64, True),  # the first row block sees most of the keys, or few
    (20, 1, 500, 500, 128, False),  # one workgroup per CU
    (32, 1, 1300, 1300, 128, False),  # the heads divide
])
def test_which_calls_are_dealt(schedule, heads_kv, group, nq, nk, d, dealt):
    schedule(heads_kv, group, nq, d, True, 4, nk)
    assert schedule.dealt == dealt
