"""How prefill launches are cut into workgroups (csrc/prefill_plan.hpp, host code without HIP), compiled and run here."""
import ctypes
import os
import random
import subprocess

import pytest

from longcontext_sqattn_paddle_amd import _native as N

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
DRIVER = r"""
#include <stdio.h>
#include <vector>
#include "prefill_plan.hpp"
int main() {
  long long off, B, Hq, Nq;
  int pq, wm, bm, sink, w8, w4, own4;
  while (scanf("%d %d %d %d %d %d %d %lld %lld %lld %lld", &pq, &wm, &bm, &sink, &w8, &w4, &own4, &off, &B, &Hq, &Nq) == 11) {
    std::vector<int32_t> a(Hq, w8), b(Hq, w4);
    sq_prefill_params p = {};
    p.p_quant = pq == 6 ? 0 : pq; p.q_offset = off; p.window_mode = wm; p.block_m = bm; p.sink = sink; p.num_heads_w = (int)Hq; p.w8 = a.data(); p.w4 = b.data();
    sq::LaunchPlan plan;
    sq::plan_launch(&p, own4 != 0, B, Hq, Nq, plan, pq == 6);   // 6: the int8 Q.K^T form of mode 0
    int w_max = w8 > w4 ? w8 : w4;
    printf("%d %d %d |", plan.waves, plan.n_work, plan.n_slots);
    for (int i = 0; i < plan.n_work; ++i) printf(" %d %d %d %d", plan.work[i].qb, plan.work[i].slot, plan.work[i].part, plan.work[i].parts);
    printf(" |");
    for (long long r = 0; r < Nq; r += 256) printf(" %d", sq::tiles_of_block(&p, r, r + 256 < Nq ? r + 256 : Nq, w_max));
    printf("\n");
  }
}
"""


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    d = tmp_path_factory.mktemp("plan")
    src, exe = d / "plan.cpp", d / "plan"
    src.write_text(DRIVER)
    subprocess.run(["g++", "-O1", "-std=c++17", "-fsanitize=undefined,address", "-fno-sanitize-recover=all", "-I", os.path.join(ROOT, "include"), "-I",
                    os.path.join(ROOT, "longcontext_sqattn_paddle_amd", "csrc"), str(src), "-o", str(exe)], check=True)

    def run(calls):
        """calls: dicts of p_quant, Nq, Hq and optionally B, offset, window = (block_m, sink, w8, w4), own4"""
        text = ""
        for c in calls:
            bm, sink, w8, w4 = c.get("window") or (128, 0, 0, 0)
            text += f"{c['p_quant']} {int(c.get('window') is not None)} {bm} {sink} {w8} {w4} {int(c.get('own4', False))} {c.get('offset', 0)} {c.get('B', 1)} {c['Hq']} {c['Nq']}\n"
        out = subprocess.run([str(exe)], input=text, capture_output=True, text=True, check=True).stdout.splitlines()
        assert len(out) == len(calls)
        plans = []
        for line in out:
            head, work, tiles = line.split("|")
            waves, n_work, n_slots = map(int, head.split())
            w = list(map(int, work.split()))
            plans.append((waves, n_slots, [tuple(w[i:i + 4]) for i in range(0, 4 * n_work, 4)], list(map(int, tiles.split()))))
        return plans

    return run


def _calls():
    rng = random.Random(7)
    calls = []
    for _ in range(3000):
        c = {"p_quant": rng.randrange(6), "Hq": rng.choice([1, 2, 3, 4, 8, 14, 28, 32, 128]), "B": rng.choice([1, 1, 1, 2, 3, 8]),
             "Nq": int(2 ** rng.uniform(0, 18)), "offset": rng.choice([0, 64 * int(2 ** rng.uniform(0, 14))])}
        kind = rng.randrange(4)
        if kind >= 2:
            bm = 64 if kind == 2 else 128
            w8 = 64 * rng.randrange(0, 40)
            c["window"] = (bm, 64 * rng.randrange(0, 10), w8, rng.choice([w8, 64 * rng.randrange(0, 400)]))
            c["offset"] = c["offset"] // 128 * 128
            c["own4"] = c["p_quant"] < 4 and rng.random() < 0.5
        calls.append(c)
    return calls


def test_every_query_block_is_covered_once(plan):
    """The work list of a split launch holds each part of each query block once, parts of a block have places of their own next
    to each other, and no part is without a tile of its (widest) head."""
    split = 0
    for c, (waves, n_slots, work, tiles) in zip(_calls(), plan(_calls())):
        assert waves in ((2,) if c.get("own4") and c["window"][0] == 64 else (4, 8)), c
        if not work:
            assert n_slots == 0
            continue
        split += 1
        assert len(work) <= 512 and c["p_quant"] != 5
        parts_of = {qb: parts for qb, _, _, parts in work}
        assert sorted((qb, part) for qb, _, part, _ in work) == [(qb, i) for qb in range(len(tiles)) for i in range(parts_of[qb])], c
        taken = set()
        for qb, slot, part, parts in work:
            assert parts == parts_of[qb] and parts <= tiles[qb], c
            if parts > 1:
                assert slot + part < n_slots and slot + part not in taken, c
                taken.add(slot + part)
        assert len(taken) == n_slots
    assert split > 300


def test_workspace_size_has_room_for_the_launch(plan):
    """The size query does not know whether the 4-bit range comes with operands of its own; it covers the launch either way."""
    part = 8 * (64 * 16 * 16 + 64 * 8 + 32 * 4)
    lib = N.lib()
    calls = [c for c in _calls() if c["B"] * c["Hq"] <= 128]
    both = [dict(c, own4=own) for c in calls for own in (False, True)]
    plans = plan(both)
    for i, c in enumerate(calls):
        Nk = c["offset"] + c["Nq"]
        w = [(ctypes.c_int32 * c["Hq"])(*[x] * c["Hq"]) for x in (c.get("window") or (0, 0, 0, 0))[2:]]
        p = N.PrefillParams(p_quant=c["p_quant"], q_offset=c["offset"])
        own = (False,)
        if c.get("window"):
            p.window_mode, p.block_m, p.sink, p.num_heads_w = N.WINDOW_SIZES, c["window"][0], c["window"][1], c["Hq"]
            p.w8, p.w4 = (ctypes.cast(x, ctypes.POINTER(ctypes.c_int32)) for x in w)
            own = (False, True)
        need = max(c["B"] * c["Hq"] * plans[2 * i + o][1] * part for o in own)
        size = lib.sq_prefill_workspace_bytes_split(c["B"], c["Hq"], c["Hq"], c["Nq"], Nk, ctypes.byref(p))
        assert size == lib.sq_prefill_workspace_bytes(c["B"], c["Hq"], Nk, 128) + need, c


def test_unsplit_choice_stands_beside_the_split(plan):
    """A call whose workspace has no room for the parts runs in the workgroups its plan found best unsplit: short calls keep
    the 128-row ones where a context in front of them brings the split on."""
    for h in (2, 4, 8):
        for n in (300, 500, 777):
            plans = plan([{"p_quant": 0, "Hq": h, "Nq": n, "offset": o} for o in (0, 256, 1024, 4096, 16384)])
            assert plans[-1][2] and all(waves == 4 for waves, _, _, _ in plans), (h, n, [waves for waves, _, _, _ in plans])


def test_a_single_half_filled_workgroup(plan):
    """Up to 128 rows a 256-row workgroup has at most four waves with rows anyway, and eight that copy the tiles: the smaller
    workgroup only where the chain of tiles is short."""
    for mode, tiles in ((0, 2), (1, 2), (2, 5), (5, 16), (6, 11)):
        for h in (1, 4, 28):
            for n in (1, 64, 100, 128):
                room = tiles - (n + 63) // 64
                got = [w for w, _, _, _ in plan([{"p_quant": mode, "Hq": h, "Nq": n, "offset": 64 * o} for o in (0, room, room + 1, 64, 2048)])]
                assert got == [4, 4, 8, 8, 8], (mode, h, n, got)
            assert all(w == 4 for w, _, _, _ in plan([{"p_quant": mode, "Hq": h, "Nq": 129, "offset": 64 * o} for o in (0, 16, 64, 2048)]))


def test_mode_4_is_not_split_where_that_only_fills_the_chip(plan):
    """Half the chip's CUs with chains of like length: split in two they run beside each other at the full chip's rate and need
    the row-maximum pass on top.  Half as many chains, or chains of unlike length, are split."""
    whole = [(4, 8192, 57344), (8, 4096, 32768), (4, 8192, 8192), (8, 4096, 131072)]
    assert not any(work for _, _, work, _ in plan([{"p_quant": 4, "Hq": h, "Nq": n, "offset": o} for h, n, o in whole]))
    split = [(4, 4096, 57344), (8, 2048, 32768), (4, 4096, 131072), (8, 4096, 0), (4, 2048, 0)]
    assert all(work for _, _, work, _ in plan([{"p_quant": 4, "Hq": h, "Nq": n, "offset": o} for h, n, o in split]))


def test_batches_of_the_pattern_tests_take_the_large_workgroups(plan):
    """The shapes whose two workgroup sizes the GPU tests compare: alone 4 waves, in the smallest batch past 512 small workgroups 8."""
    for mode in (0, 1, 2, 5):
        for n, offset in ((777, 0), (1536, 0), (512, 2048)):
            for window in (None, (64, 64, 128, 256), (64, 0, 64, 64)):
                copies = 512 // (4 * ((n + 127) // 128)) + 1
                alone, many = plan([{"p_quant": mode, "Hq": 4, "Nq": n, "offset": offset, "window": window, "B": b} for b in (1, copies)])
                assert alone[0] == 4 and many[0] == 8, (mode, n, window)


def test_windows_without_a_sink_are_split_in_the_grid_modes_only(plan):
    """The parts of modes 0 and 6 start from the row's scores of tile 0, which such windows do not reach."""
    for mode, sink, split in ((0, 64, True), (6, 64, True), (0, 0, False), (6, 0, False), (1, 0, True), (2, 0, True), (4, 0, True)):
        (_, _, work, _), = plan([{"p_quant": mode, "Hq": 2, "Nq": 4096, "window": (64, sink, 1024, 2048)}])
        assert bool(work) is split, (mode, sink)


def test_split_blocks_see_all_of_the_first_tile(plan):
    """No row of a block with parts sits among the first 64 keys."""
    calls = _calls()
    for c, (_, _, work, _) in zip(calls, plan(calls)):
        assert all(c["offset"] + 256 * qb >= 64 for qb, _, _, parts in work if parts > 1), c


def test_value_tiles_beside_the_row_maximum_pass(tmp_path):
    """The calls of the GPU test of that path take it, in one, two and ten rounds; short chunks behind long contexts keep the launch of
    their own."""
    src, exe = tmp_path / "beside.cpp", tmp_path / "beside"
    src.write_text(r"""
#include <stdio.h>
#include "prefill_plan.hpp"
int main() {
  long long B, Hq, Hkv, Nq, off;
  int pq;
  while (scanf("%d %lld %lld %lld %lld %lld", &pq, &B, &Hq, &Hkv, &Nq, &off) == 6) {
    sq_prefill_params p = {};
    p.p_quant = pq; p.q_offset = off; p.block_m = 128;
    sq::LaunchPlan plan;
    sq::plan_launch(&p, false, B, Hq, Nq, plan);
    const long long tiles = B * Hkv * ((off + Nq + 63) / 64), idle = B * Hq * ((Nq + 255) / 256);
    printf("%d %lld\n", plan.n_work > 0 ? 1 + sq::prep_beside_pass(plan.share, tiles, idle) : 0, (tiles + 2 * idle - 1) / (2 * idle));
  }
}
""")
    subprocess.run(["g++", "-O1", "-std=c++17", "-I", os.path.join(ROOT, "include"), "-I", os.path.join(ROOT, "longcontext_sqattn_paddle_amd", "csrc"),
                    str(src), "-o", str(exe)], check=True)
    calls = {(2, 2, 4, 2, 2048, 0): (2, 1), (3, 2, 4, 2, 2048, 0): (2, 1), (2, 1, 8, 8, 2048, 0): (2, 2), (2, 2, 4, 4, 2000, 0): (2, 2), (3, 2, 4, 4, 2000, 0): (2, 2),
             (2, 1, 14, 2, 300, 2048): (2, 2), (1, 1, 28, 4, 512, 16384): (2, 10), (1, 1, 28, 4, 64, 16384): (1, 19), (2, 1, 3, 1, 200, 3072): (1, 9)}
    text = "".join(" ".join(map(str, c)) + "\n" for c in calls)
    out = subprocess.run([str(exe)], input=text, capture_output=True, text=True, check=True).stdout.split()
    assert [tuple(map(int, out[i:i + 2])) for i in range(0, len(out), 2)] == list(calls.values())
