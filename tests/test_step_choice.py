"""The one-console-per-wave step kernels without a GPU: the rules that choose a
batch's kernel (nesle_amd/csrc/nes_choice.h, compiled alone) -- images whose
flow runs past $FFFF, the choice from step to step -- and where their dispatch tables may lie."""

from __future__ import annotations

import ctypes
import os
import shutil
import subprocess

import numpy as np
import pytest

from nesle_amd import build

CXX = os.environ.get("CXX") or shutil.which("g++") or shutil.which("clang++")
pytestmark = pytest.mark.skipif(CXX is None, reason="no host C++ compiler")

SHIM = r"""
#include "nes_choice.h"
using namespace nesle;
extern "C" {
int t_closed_end(const std::uint8_t* prg, std::size_t size) { return closed_end(prg, size); }
// `steps` steps of a program that goes over the limit in the per-wave steps
// for which over[step] is set; the kernel of each into out.
void t_choices(const std::uint8_t* over, std::uint8_t* out, std::uint32_t steps) {
    StepChoice c{};
    for (std::uint32_t k = 0; k < steps; ++k) {
        c.now = c.next;
        if (c.now == 0)
            for (std::uint32_t i = 0; i < kGeneralSlots; ++i) c.over[i] = over[k] && i == k % kGeneralSlots;
        out[k] = static_cast<std::uint8_t>(c.now);
        choice_update(c);
    }
}
int t_over(std::uint32_t n, std::uint32_t trips, std::uint32_t jumps, std::uint32_t frames) {
    return over_limit(general_limit(n), trips, jumps, frames, 341 * 262);
}
}
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    work = tmp_path_factory.mktemp("choice")
    (work / "shim.cpp").write_text(SHIM)
    subprocess.run([CXX, "-std=c++17", "-O1", "-shared", "-fPIC", f"-I{build.CSRC}", str(work / "shim.cpp"), "-o",
                    str(work / "shim.so")], check=True, capture_output=True, text=True)
    L = ctypes.CDLL(str(work / "shim.so"))
    L.t_closed_end.argtypes = [ctypes.c_char_p, ctypes.c_size_t]
    L.t_choices.argtypes = [ctypes.c_char_p, ctypes.c_char_p, ctypes.c_uint32]
    return L


# Lengths of the official opcodes, one row per high digit (0: illegal), and
# those that do not go on to the next instruction (BRK, JSR, RTI, JMP, RTS).
LENGTHS = [int(c) for row in (
    "1200022012100330", "2200022013000330", "3200222012103330", "2200022013000330",
    "1200022012103330", "2200022013000330", "1200022012103330", "2200022013000330",
    "0200222010103330", "2200222013100300", "2220222012103330", "2200222013103330",
    "2200222012103330", "2200022013000330", "2200222012103330", "2200022013000330") for c in row]
LEAVES = {0x00, 0x20, 0x40, 0x4C, 0x60, 0x6C}


def runs_past_the_end(prg: bytes) -> bool:
    """Walks the flow from every start in the last bytes below $FFFA."""
    for at in range(len(prg) - 26, len(prg) - 6):
        while at < len(prg):
            op = prg[at]
            if LENGTHS[op] == 0:
                break
            if at + LENGTHS[op] > len(prg):
                return True
            if op in LEAVES:
                break
            at += LENGTHS[op]
    return False


@pytest.mark.parametrize("tail,open_end", [
    ([0xEA] * 9, False),                                                     # NOPs end at $FFFF
    ([0xEA] * 8 + [0xAD], True),                                             # LDA abs at $FFFF
    ([0xAD, 0x02, 0x03] + [0xEA] * 5 + [0xAD], True),                        # over $FFF7-$FFF9, no opcodes there
    ([0x8D, 0x02, 0x03] + [0xEA] * 5 + [0xA5], True),
    ([0x4C, 0x02, 0x03] + [0xEA] * 5 + [0xAD], False),                       # a jump at $FFF7 goes nowhere else
    ([0x02, 0x02, 0x02] + [0xEA] * 5 + [0xAD], False),                       # nothing falls into the vectors
    ([0xA5, 0x02, 0x02] + [0xEA] * 5 + [0xAD], False),                       # two bytes end at $FFF8
])
def test_images_whose_flow_runs_past_the_end(lib, tail, open_end):
    """Tails from $FFF7 on, the rest of the image illegal opcodes."""
    prg = bytes([0x02] * (32768 - len(tail)) + tail)
    assert runs_past_the_end(prg) == open_end
    assert bool(lib.t_closed_end(prg, len(prg))) == (not open_end)


def test_random_images_agree_with_a_walk_of_the_flow(lib):
    """Random tails, of all bytes and of few illegal ones, both image sizes."""
    rng = np.random.default_rng(5)
    legal = np.array([op for op in range(256) if LENGTHS[op] and op not in LEAVES], dtype=np.uint8)
    seen = {True: 0, False: 0}
    for k in range(4000):
        size = 16384 if k % 2 else 32768
        tail = rng.integers(0, 256, 32).astype(np.uint8)
        mostly = rng.random(32) < (0.0, 0.5, 0.9)[k % 3]
        tail[mostly] = rng.choice(legal, int(mostly.sum()))
        prg = bytes(size - 32) + bytes(tail)
        want = runs_past_the_end(prg)
        seen[want] += 1
        assert bool(lib.t_closed_end(prg, size)) == (not want), tail.tobytes().hex()
    assert min(seen.values()) > 200


def kernels(lib, over: list[bool]) -> list[int]:
    """0 (one console per wave) or 1 (the lane kernel) for each step."""
    out = ctypes.create_string_buffer(len(over))
    lib.t_choices(bytes(over), out, len(over))
    return list(out.raw)


def test_kernel_of_each_step(lib):
    """Steps within the limit stay; a step over it is followed by 64 lane steps."""
    assert kernels(lib, [False] * 200) == [0] * 200
    # One bad step among good ones, wherever it falls.
    for at in (0, 1, 17):
        over = [k == at for k in range(at + 70)]
        assert kernels(lib, over) == [0] * (at + 1) + [1] * 64 + [0] * 5


def test_trials_of_a_program_that_stays_over_the_limit_grow_rare(lib):
    """One step is tried after 64, 256, 1,024 and from then on 4,096 lane steps."""
    got = kernels(lib, [True] * 20000)
    tried = [k for k, kernel in enumerate(got) if kernel == 0]
    assert tried[:4] == [0, 65, 322, 1347]
    assert set(np.diff(tried[3:])) == {4097}
    # At 32,768 consoles a trial takes some 430 ms, a lane step 17: under 1 %.
    assert (len(tried) - 4) * 430 < 0.01 * (20000 - 1347) * 17


def test_trials_start_over_after_a_run_of_good_steps(lib):
    """Twice over the limit in a row: the stays are 64 and 256; the third one
    is 64 again only after 1,024 good steps, the length it would have had."""
    for good, third in ((1023, 1024), (1024, 64)):
        first = 1 + 64 + 1 + 256            # both bad steps and their stays
        over = [k in (0, 65, first + good) for k in range(first + good + 1200)]
        got = kernels(lib, over)
        assert got[:first + good + 1] == [0] + [1] * 64 + [0] + [1] * 256 + [0] * (good + 1)
        rest = got[first + good + 1:]
        assert rest[:third] == [1] * third and rest[third] == 0


def limit(lib, n: int, busy: float) -> int:
    """Trips a frame allowed to a program that idles the rest of its frame."""
    jumps = round((1 - busy) * 341 * 262 * 4 / 9)
    return next(t for t in range(100000) if lib.t_over(n, 4 * t + 4, jumps, 4))


def test_limit_falls_as_the_batch_grows_and_the_program_idles(lib):
    assert [limit(lib, n, 1.0) for n in (4096, 8192, 16384, 32768)] == [1144, 539, 267, 63]
    assert [limit(lib, n, 0.3) for n in (4096, 8192, 16384, 32768)] == [347, 164, 81, 19]
    sizes = [1, 64, 1000, 2457, 2458, 4096, 8192, 20000, 32768]
    for busy in (0.0, 0.1, 0.5, 1.0):
        got = [limit(lib, n, busy) for n in sizes]
        assert got == sorted(got, reverse=True)
    # Jumps beyond the frames (a console that starts inside one) are no credit.
    assert not lib.t_over(1, 10, 1 << 20, 1) and lib.t_over(1, 11, 1 << 20, 1)


# Measured, us per step of four frames: a program that waits for its NMI, runs
# `work` turns of a 26-cycle loop and reads $4015 `reads` times in one of 9
# cycles, with one console per wave and by the lane kernel.
MEASURED = [
    (1000, 4, 0, 52, 207), (1000, 4, 20, 188, 323), (1000, 4, 60, 456, 562), (1000, 4, 200, 1390, 1380),
    (1000, 4, 500, 3380, 3143), (1000, 60, 0, 173, 1093), (1000, 60, 20, 306, 1189), (1000, 60, 60, 569, 1409),
    (1000, 60, 200, 1497, 2211), (1000, 60, 500, 3489, 3995), (1000, 200, 0, 489, 3337), (1000, 200, 20, 601, 3294),
    (1000, 200, 60, 861, 3560), (1000, 200, 200, 1783, 4353), (1000, 200, 500, 3787, 6107), (4096, 4, 0, 94, 180),
    (4096, 4, 20, 341, 300), (4096, 4, 60, 834, 544), (4096, 4, 200, 2541, 1349), (4096, 4, 500, 6056, 3089),
    (4096, 60, 0, 228, 1076), (4096, 60, 20, 472, 1163), (4096, 60, 60, 960, 1399), (4096, 60, 200, 2593, 2211),
    (4096, 60, 500, 6185, 3945), (4096, 200, 0, 547, 3290), (4096, 200, 20, 788, 3288), (4096, 200, 60, 1274, 3530),
    (4096, 200, 200, 2896, 4332), (4096, 200, 500, 6600, 6081), (8192, 4, 0, 157, 223), (8192, 4, 20, 612, 347),
    (8192, 4, 60, 1512, 581), (8192, 4, 200, 4720, 1406), (8192, 4, 500, 11332, 3191), (8192, 60, 0, 310, 1134),
    (8192, 60, 20, 752, 1216), (8192, 60, 60, 1645, 1436), (8192, 60, 200, 4732, 2286), (8192, 60, 500, 11368, 4010),
    (8192, 200, 0, 698, 3307), (8192, 200, 20, 1116, 3410), (8192, 200, 60, 2001, 3610), (8192, 200, 200, 5121, 4394),
    (8192, 200, 500, 11992, 6166), (16384, 4, 0, 278, 178), (16384, 4, 20, 1175, 332), (16384, 4, 60, 2958, 635),
    (16384, 4, 200, 9235, 1659), (16384, 4, 500, 22497, 3888), (16384, 60, 0, 579, 1230), (16384, 60, 20, 1448, 1378),
    (16384, 60, 60, 3243, 1673), (16384, 60, 200, 9420, 2708), (16384, 60, 500, 22684, 4904),
    (16384, 200, 0, 1352, 3837), (16384, 200, 20, 2179, 3961), (16384, 200, 60, 3924, 4300),
    (16384, 200, 200, 10134, 5382), (16384, 200, 500, 23594, 7494), (32768, 4, 0, 535, 179),
    (32768, 4, 20, 2299, 327), (32768, 4, 60, 5854, 616), (32768, 4, 200, 18328, 1612), (32768, 4, 500, 44783, 3737),
    (32768, 60, 0, 1120, 1232), (32768, 60, 20, 2865, 1384), (32768, 60, 60, 6446, 1685),
    (32768, 60, 200, 18760, 2665), (32768, 60, 500, 45217, 4803), (32768, 200, 0, 2652, 3854),
    (32768, 200, 20, 4313, 3994), (32768, 200, 60, 7812, 4305), (32768, 200, 200, 20148, 5282),
    (32768, 200, 500, 46848, 7427),
]


def test_limit_picks_the_quicker_kernel(lib):
    """Wherever one of the two takes at least 1.25 times as long (nearer than
    that the rule, which knows cycles and not instructions, misses four)."""
    for n, work, reads, wave_us, lane_us in MEASURED:
        if max(wave_us, lane_us) < 1.25 * min(wave_us, lane_us):
            continue
        cycles = 26 * work + 9 * reads + 25                # with the NMI entry and its return
        jumps = 4 * (29781 - cycles) // 3
        over = lib.t_over(n, 4 * (reads + 5), jumps, 4)    # five trips besides the reads: NMI, four waits
        assert bool(over) == (wave_us > lane_us), (n, work, reads)


WAVE = build.CSRC / "nes_wave.h"


def enter(table: int, solo: bool) -> dict | None:
    """The assembly's own test of where its dispatch table lies, followed line
    by line for a table at that address: the registers with which the block is
    entered, or None where nothing runs in it."""
    text = WAVE.read_text()
    at = text.index("  s_mov_b32 s[rTab], s[rJ]")
    lines = [ln.split(";")[0].strip() for ln in text[at:text.index(".Lw%=_end:", at)].splitlines()]
    reg = {"rJ": table & 0xFFFFFFFF}
    scc, skip, k = 0, False, 0

    def value(x: str) -> int:
        return reg[x[2:-1]] if x.startswith("s[") else int(x, 0)

    while True:
        op, _, rest = lines[k].partition(" ")
        a = [x.strip() for x in rest.split(",")]
        k += 1
        if op == ".if":
            assert a == ["SOLO"]
            skip = not solo
        elif op == ".endif":
            skip = False
        elif skip or not op or op == "UNPACK" or (op.endswith(":") and op != ".Lw%=_start:"):
            continue
        elif op == "PACK":
            return None
        elif op == ".Lw%=_start:":
            return reg
        elif op == "s_mov_b32":
            reg[a[0][2:-1]] = value(a[1])
        elif op == "s_sub_u32":
            reg[a[0][2:-1]] = (value(a[1]) - value(a[2])) & 0xFFFFFFFF
        elif op == "s_and_b32":
            reg[a[0][2:-1]] = value(a[1]) & value(a[2])
            scc = int(reg[a[0][2:-1]] != 0)
        elif op == "s_cmp_eq_u32":
            scc = int(value(a[0]) == value(a[1]))
        elif op in ("s_cbranch_scc0", "s_cbranch_scc1"):
            if scc == int(op[-1]):
                k = lines.index(a[0] + ":")
        else:
            raise AssertionError(f"unexpected line: {lines[k - 1]}")


@pytest.mark.parametrize("solo", [True, False])
@pytest.mark.parametrize("table", [0x7F0012340000, 0x7F0000010000, 0x7F00FFFF0000, 0x7F0000000000, 0x7F0012340100,
                                   0x7F0000000100])
def test_dispatch_tables_are_reached_by_their_low_half(table, solo):
    """A jump replaces only the low 32 bits of the table's address, so the
    solo form's exit table (64 KB below) must share its high ones; and the
    table must be aligned to its 64 KB.  Elsewhere nothing runs in the block."""
    reg = enter(table, solo)
    fits = table % 0x10000 == 0 and (not solo or (table - 0x10000) >> 32 == table >> 32)
    assert (reg is not None) == fits
    if reg is not None:
        assert reg["rTab"] == reg["rQ"] == table & 0xFFFFFFFF
        if solo:
            assert (table >> 32 << 32 | reg["rExit"]) == table - 0x10000
