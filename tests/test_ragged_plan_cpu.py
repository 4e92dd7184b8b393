"""The one-workgroup ragged plan (ragged_plan_small), compiled for the host and
run with its threads taken in several orders: what one thread reads of
another's must lie behind a barrier, whatever wave or order the threads run
in.  Checked: class counts, first slots, descriptors, matrices per descriptor,
the invalid count, and that every class's slots hold its matrices."""
import os
import re
import subprocess

import numpy as np
import pytest

from tests.conftest import ROOT

CSRC = os.path.join(ROOT, "matrixinversion_amd", "csrc")

DRIVER = r"""
#include <cstdio>
#include <cstring>
int main(int argc, char** argv) {
  const int64_t batch = atoll(argv[1]);
  const int mode = atoi(argv[2]);
  std::vector<int> ns(batch), ws(lub::RaggedWs::HEADER, -777), order(lub::kSmallPlanThreads);
  std::vector<int64_t> offs(batch), poffs(batch), so(batch, -1), sp(batch, -1);
  if (fread(ns.data(), 4, batch, stdin) != size_t(batch)) return 2;
  for (int64_t i = 0; i < batch; ++i) { offs[i] = 7 * i; poffs[i] = 3 * i; }
  lub::RaggedTuning tune;
  for (int n = 0; n <= 32; ++n) { tune.layout[n] = n <= 12; tune.grab[n] = n <= 12 ? 1 : 8; }
  const int count = int(order.size());
  for (int i = 0; i < count; ++i) order[i] = mode == 0 ? i : mode == 1 ? count - 1 - i : (i * 389 + 5) % count;
  emu::run(order, [&] { lub::ragged_plan_small(ns.data(), offs.data(), poffs.data(), batch, ws.data(), tune, so.data(),
                                               sp.data()); });
  fwrite(ws.data(), 4, ws.size(), stdout);
  fwrite(so.data(), 8, batch, stdout);
  fwrite(sp.data(), 8, batch, stdout);
}
"""


def _block(text, start):
    """The declaration that begins at `start`, to the end of its braces."""
    at = text.index(start)
    depth, i = 0, text.index("{", at)
    while True:
        depth += {"{": 1, "}": -1}.get(text[i], 0)
        i += 1
        if depth == 0:
            return text[at:i] + (";" if text[at:at + 6] == "struct" else "") + "\n"


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    head = open(os.path.join(CSRC, "lu_ragged.hpp")).read()
    unit = open(os.path.join(CSRC, "lub_ragged.hip")).read()
    parts = [_block(head, "struct RaggedTuning"), _block(head, "struct RaggedWs")]
    parts += re.findall(r"^constexpr int kRagged(?:QuadMaxN|MaxPer) = .*$", head, flags=re.M)
    parts += [_block(head, "__host__ __device__ constexpr int ragged_grab_limit"),
              _block(head, "__host__ __device__ constexpr int ragged_mpw")]
    table = re.search(r"__device__[\w ]* void ragged_class_table", unit).group(0)
    parts += ["constexpr int kWave = 64;", _block(unit, table)]
    parts += re.findall(r"^constexpr \w+ kSmallPlan\w+ = .*$", unit, flags=re.M)
    parts += [_block(unit, "__global__ __launch_bounds__(kSmallPlanThreads) void ragged_plan_small")]
    d = tmp_path_factory.mktemp("plan")
    src, exe = d / "plan.cpp", d / "plan"
    src.write_text('#include "block_emulator.hpp"\nnamespace lub {\n' + "\n".join(parts) + "\n}\n" + DRIVER)
    subprocess.run(["g++", "-std=c++20", "-O1", "-Wno-unknown-pragmas", "-I", os.path.join(ROOT, "tests"), str(src),
                    "-o", str(exe)], check=True)
    return str(exe)


@pytest.mark.parametrize("mode", [0, 1, 2])
@pytest.mark.parametrize("batch,lo,hi", [(2049, 1, 32), (3000, 4, 32), (16384, 1, 32), (16384, 32, 32), (5000, 1, 3)])
def test_small_plan_in_any_thread_order(plan, batch, lo, hi, mode):
    rng = np.random.RandomState(batch + lo)
    ns = rng.randint(lo, hi + 1, batch).astype(np.int32)
    ns[rng.permutation(batch)[:batch // 20]] = rng.choice([0, -2, 33, 4000], batch // 20)
    out = subprocess.run([plan, str(batch), str(mode)], input=ns.tobytes(), stdout=subprocess.PIPE, check=True).stdout
    ws = np.frombuffer(out, np.int32, 384)
    so, sp = np.frombuffer(out, np.int64, 2 * batch, 384 * 4).reshape(2, batch)
    counts = {n: int((ns == n).sum()) for n in range(1, 33)}
    mpw = {n: 16 if n <= 12 else 4 for n in counts}
    tiles = sum(-(-counts[n] // mpw[n]) for n in counts)
    slot = desc = 0
    for n in range(32, 0, -1):  # largest first
        limit = max(1, tiles // (2048 if n <= 16 else 4096))
        per = mpw[n] * min(1 if n <= 12 else 8, limit)
        assert (ws[n], ws[128 + n], ws[192 + n], ws[320 + n]) == (counts[n], slot, desc, (n <= 12) | per << 8), n
        where = np.flatnonzero(ns == n)
        assert np.array_equal(np.sort(so[slot:slot + counts[n]]), 7 * where)
        assert np.array_equal(so[slot:slot + counts[n]] // 7, sp[slot:slot + counts[n]] // 3)
        slot += counts[n]
        desc += -(-counts[n] // per)
    assert ws[192] == desc and ws[258] == batch - slot
