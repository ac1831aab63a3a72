"""Blocks of a causal walk in parts, on the host: a plan's jobs are every part of every block once, longest first; plans are searched
for once; the libraries report the room their plans take."""
import ctypes
import os
import random
import subprocess

import pytest

from attention_autotuner_amd.arch import MI355X
from attention_autotuner_amd.autotuner import codegen, gfx950_space, library, runtime

MOST_PARTS, MOST_JOBS, ORDER_BYTES = 4, 256, 512
RULE = [(op, d, c) for op in ("ret", "ret_bwd") for d in sorted(gfx950_space.RET_RULE) for c in gfx950_space.rule_ret_configs(op, *d)]

SOURCE = r"""
#include <hip/hip_runtime.h>
#include "kernels/utils/block_parts.h"
extern "C" int plan(long heads, int T, const int* walks, double tile_us, int waves, int blocks_per_cu, int rounds, size_t slot, int* split, int* parts, int* jobs) {
  const auto walk = [=](int t) { return walks[t]; };
  const aat::PartsPlan p = aat::plan_parts(heads, T, walk, aat::PartsCost{tile_us, waves, blocks_per_cu, rounds, slot});
  *split = p.split;
  *parts = p.parts;
  return aat::each_job(T, p, walk, [&](int n, int rank, int part) { jobs[n] = 8 * rank + (part < 0 ? 0 : part); });
}
extern "C" void share(int part, int parts, int* begin, int* end) { aat::part_range(aat::PartId{0, 0, part, parts, 0}, *begin, *end); }
extern "C" void walks(int rows, int T, int Br, int Bc, int Seq_q, int Seq_k, int* out) {
  for (int t = 0; t < T; ++t) out[t] = rows ? aat::row_walk(t, Br, Bc, Seq_q, Seq_k) : aat::col_walk(t, Br, Bc, Seq_q, Seq_k);
}
// how often plans are searched for where the problems (heads, Seq_q, Seq_k, blocks per CU) come in this order, by one launch's memory
extern "C" int searches(const int* problems, int n) {
  static aat::PlanMemory known;
  int count = 0;
  for (int i = 0; i < n; ++i) {
    const int* p = problems + 4 * i;
    const aat::PartsPlan got = known.get(p[0], p[1], p[2], p[3], [&] { ++count; return aat::PartsPlan{p[1] / 64, 1 + p[2] / 64}; });
    if (got.split != p[1] / 64 || got.parts != 1 + p[2] / 64) return -1;
  }
  return count;
}
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    work = tmp_path_factory.mktemp("parts")
    src, out = str(work / "plan.hip"), str(work / "plan.so")
    with open(src, "w") as f:
        f.write(SOURCE)
    subprocess.run(codegen.hipcc_command(src, out, MI355X()), check=True, capture_output=True, cwd=str(work))
    return ctypes.CDLL(out)


def _walks(rows, br, bc, seq_q, seq_k):
    """Tiles a block walks below the diagonal kv <= q + seq_k - seq_q, the longest block first."""
    diag = seq_k - seq_q
    if rows:
        firsts = range((-(-seq_q // br) - 1) * br, -1, -br)
        return [max(0, min(seq_k // bc, (min(q0 + br, seq_q) - 1 + diag) // bc + 1)) for q0 in firsts]
    return [max(0, seq_q // bc - max(0, k0 - diag) // bc) for k0 in range(0, seq_k, br)]


def test_the_jobs_of_a_plan_are_complete_and_longest_first(lib):
    rng = random.Random(5)
    cut = 0
    for _ in range(150):
        br, bc, waves = rng.choice(((128, 64, 4), (64, 64, 2), (64, 32, 2), (128, 32, 4)))
        sq, sk = 64 * rng.randint(1, 64), 64 * rng.randint(1, 64)
        heads, rows, per_cu = rng.randint(1, 32), rng.randint(0, 1), rng.choice((1, 2, 4))
        cols, width = rng.choice(((64, 128), (128, 256), (256, 512), (256, 768), (512, 768)))
        want = _walks(bool(rows), br, bc, sq, sk)
        T = len(want)
        got = (ctypes.c_int * T)()
        lib.walks(rows, T, br, bc, sq, sk, got)
        assert list(got) == want, (rows, br, bc, sq, sk)
        tile, slot = 2.0 * br * bc * width / 4.5e6, br * cols * 4
        c_split, c_parts, jobs = ctypes.c_int(), ctypes.c_int(), (ctypes.c_int * (T * MOST_PARTS))()
        n = lib.plan(ctypes.c_long(heads), T, got, ctypes.c_double(tile), waves, per_cu, br * cols // (256 * waves) // 4, ctypes.c_size_t(slot),
                     ctypes.byref(c_split), ctypes.byref(c_parts), jobs)
        split, parts = c_split.value, c_parts.value
        assert sorted(jobs[:n]) == sorted([8 * t + p for t in range(split) for p in range(parts)] + [8 * t for t in range(split, T)])
        lengths = [want[j >> 3] / (parts if j >> 3 < split else 1) for j in jobs[:n]]
        assert all(a >= b - 1e-9 for a, b in zip(lengths, lengths[1:]))
        assert split == 0 or (n <= MOST_JOBS and want[split - 1] >= 2 * parts)
        cut += split > 0
    assert 20 <= cut <= 130


@pytest.mark.parametrize("op", ["ret", "ret_bwd"])
def test_the_libraries_report_the_room_of_their_parts(op):
    rng, cut = random.Random(7), 0
    for _, d, cfg in (r for r in RULE if r[0] == op):
        loaded = library.load(codegen.compile_config(cfg, MI355X(), timeout=600), op)
        for _ in range(40):
            b, h, sq = rng.randint(1, 4), rng.choice((1, 2, 3, 4, 8, 12)), 64 * rng.randint(1, 48)
            sk = rng.choice((sq, 64 * rng.randint(1, 48)))
            problem, heads = (b, h, sq, sk), b * h
            least, most = loaded.decay_workspace_size(*problem, 0), loaded.decay_workspace_size(*problem, ctypes.c_size_t(-1).value)
            ds = 2 * b * h * sq * sk if loaded.workspace_size(*problem) >= 2 * b * h * sq * sk and getattr(cfg, "ds_rows", 0) else 0
            assert least == loaded.workspace_size(*problem) - ds and most >= loaded.workspace_size(*problem)
            # counts are whole units of 256 bytes, each launch has an order, slots hold the resident rows of a block in fp32
            for stored in {0, ds}:
                total = loaded.decay_workspace_size(*problem, max(ds, 1 << 40)) if stored == ds else loaded.decay_workspace_size(*problem, ds - 1)
                room = total - least - stored
                if room > 0:
                    launches = 1 if op == "ret" else 3
                    assert room % 256 == 0 and room > launches * ORDER_BYTES + heads * 2 * 64 * cfg.Kd * 4
                    assert loaded.decay_workspace_size(*problem, max(stored, room)) in (total, least + ds + room)
                    cut += 1
        assert loaded.decay_workspace_size(1, 1, 16, 16, 1 << 40) == loaded.workspace_size(1, 1, 16, 16)      # no length it takes
    assert cut > 40


# Problems measured whole and in the parts an estimate without the exchange's cost and the XCDs' shares of the jobs picked
@pytest.mark.parametrize("op,dqk,dv,b,h,s,pays", [
    ("ret_bwd", 192, 192, 1, 8, 832, False),       # 69 us whole, 90 in parts
    ("ret_bwd", 256, 256, 4, 8, 1088, False),
    ("ret", 256, 512, 1, 4, 512, False),           # 28.6, 35.6
    ("ret", 256, 512, 5, 4, 1344, False),          # 64.4, 87.8
    ("ret", 192, 192, 1, 10, 3008, False),         # 73.9, 95.7
    ("ret", 128, 128, 1, 4, 4096, True),           # 80, 47
    ("ret_bwd", 128, 128, 1, 4, 4096, True),       # 238, 173
    ("ret_bwd", 64, 64, 1, 2, 4096, True),
    ("ret", 256, 512, 1, 8, 2048, True),           # 101, 64
    ("ret_bwd", 256, 512, 2, 8, 2112, True)])      # 257, 211
def test_only_what_pays_is_cut(op, dqk, dv, b, h, s, pays):
    cfg = gfx950_space.rule_ret_config(op, dqk, dv, b, h, s, s, True)
    loaded = library.load(codegen.compile_config(cfg, MI355X(), timeout=600), op)
    whole = loaded.workspace_size(b, h, s, s)
    assert (loaded.decay_workspace_size(b, h, s, s, 1 << 40) > whole) == pays


def test_a_library_without_the_question_is_asked_for_its_workspace_size():
    class Old:
        pass
    cfg = next(c for op, d, c in RULE if op == "ret_bwd" and c.ds_rows)
    assert runtime._provided(Old(), cfg, 4096, 1, 8, 512, 512, True) == 4096

    class New:
        def decay_workspace_size(self, *problem_and_limit):
            assert problem_and_limit == (1, 8, 512, 512, runtime.MAX_DS_BYTES)
            return 9999
    assert runtime._provided(New(), cfg, 4096, 1, 8, 512, 512, True) == 9999
    assert runtime._provided(New(), cfg, 4096, 1, 8, 512, 512, False) == 4096


def test_shares_cover_the_walk(lib):
    for first in (0, 3, 17):
        for n in range(0, 70):
            for parts in (1, 2, 3, 4):
                begin, end, at = ctypes.c_int(), ctypes.c_int(), first
                for part in range(parts):
                    begin.value, end.value = first, first + n
                    lib.share(part, parts, ctypes.byref(begin), ctypes.byref(end))
                    assert begin.value == at and end.value - begin.value in (n // parts, n // parts + 1), (first, n, parts, part)
                    at = end.value
                assert at == first + n
    begin, end = ctypes.c_int(5), ctypes.c_int(3)                       # an empty walk
    lib.share(1, 2, ctypes.byref(begin), ctypes.byref(end))
    assert begin.value == end.value == 5


def test_lengths_in_turn_are_searched_for_once(lib):
    lengths = [64 * i for i in range(1, 65)]
    problems = [(h, s, s, 1) for _ in range(3) for s in lengths for h in (8, 32)] + [(8, 64, 128, 1), (8, 64, 128, 2), (8, 64, 128, 1)] * 5
    flat = (ctypes.c_int * (4 * len(problems)))(*[x for p in problems for x in p])
    assert 128 + 2 <= lib.searches(flat, len(problems)) <= 128 + 2 + 16          # sets of four: a few problems push each other out


@pytest.mark.parametrize("op", ["ret", "ret_bwd"])
def test_decay_calls_touch_thread_storage_of_their_library(op):
    """... which is what keeps torch's own accesses off glibc's slow path on the host (utils/host_launch.h)."""
    cfg = next(c for o, d, c in RULE if o == op and d == (64, 64))
    segments = subprocess.run(["readelf", "-lW", codegen.compile_config(cfg, MI355X(), timeout=600)], check=True, capture_output=True, text=True).stdout
    assert " TLS " in segments
    entry = codegen.render(cfg).split("hipError_t launch_decay(")[1].split("\n}")[0]
    assert "aat::touch_thread_storage();" in entry
