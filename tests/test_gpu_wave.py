"""The one-console-per-wave step kernels (nes_step_wave.hip, nes_step_solo.hip),
which run plain steps of up to 32,768 consoles, and the choice between them and
the lane kernel.  A statistics step runs the lane kernel, which the oracle
tests pin, so three batches -- stepped by these kernels, by the lane kernel
without statistics and by it with them -- must agree in every byte: over programs that take each
side path (I/O, PRG RAM, code in RAM, stack and address wraps, illegal
opcodes, OAM DMA from every kind of page, the idle loop) and over sizes at the
edges of the workgroup shapes.  Programs that run into and over the vectors
are compared with the oracle itself."""

from __future__ import annotations

import os
import re
import shutil
import subprocess
import sys
from pathlib import Path

import numpy as np
import pytest

from nesle_amd import abi, build, synthrom
from oracle import oracle as O
from tests.helpers import first_diff, masks_for, say
from tests.kat_roms import nrom_bytes
from tests.test_gpu_features import address_wrap_rom, feature_rom, io_corner_rom, oam_rom, stack_wrap_rom
from tests.test_gpu_idle import idle_rom

def wait_rom() -> bytes:
    """Loops that wait for PPUSTATUS flags, in every form the kernel skips and
    some it must not: LDA or BIT, with and without AND #, across a page, with
    the read's open-bus bits in play, a loop that falls through at once, one
    whose branch leads elsewhere."""
    def at(addr, *code):
        return addr, list(code)

    parts = dict([
        at(0x8000, 0x78, 0xA2, 0xFF, 0x9A, 0xA9, 0x80, 0x8D, 0x00, 0x20, 0xA9, 0x18, 0x8D, 0x01, 0x20, 0x4C, 0x00, 0x81),
        at(0x8100, 0xAD, 0x02, 0x20, 0x10, 0xFB, 0xE6, 0x20, 0x4C, 0xFC, 0x82),              # LDA; BPL (vblank)
        at(0x82FC, 0x2C, 0x02, 0x20, 0x70, 0xFB, 0xE6, 0x21, 0x4C, 0xFB, 0x83),              # BIT; BVS, over a page
        at(0x83FB, 0x2C, 0x02, 0x20, 0x50, 0xFB, 0xE6, 0x22, 0x4C, 0x00, 0x85),              # BIT; BVC, over a page
        at(0x8500, 0xAD, 0x02, 0x20, 0x29, 0x40, 0xD0, 0xF9, 0xE6, 0x23, 0x4C, 0xF9, 0x86),  # LDA; AND #$40; BNE
        at(0x86F9, 0xAD, 0x02, 0x20, 0x29, 0x40, 0xF0, 0xF9, 0xE6, 0x24, 0x85, 0x25),        # ... BEQ, over a page
        at(0x8704, 0x8E, 0x05, 0x20, 0xAD, 0x02, 0x20, 0x29, 0x1F, 0x85, 0x26, 0xCA),        # open bus = X
        at(0x870F, 0xAD, 0x02, 0x20, 0x30, 0xFB, 0x2C, 0x02, 0x20, 0x90, 0x02, 0xE6, 0x27),  # BMI; BCC elsewhere
        at(0x871B, 0x2C, 0x02, 0x20, 0x29, 0xFF, 0xD0, 0xF9, 0x4C, 0x00, 0x81),              # BIT; AND #; BNE
        at(0x9000, 0x48, 0xE6, 0x10, 0xA5, 0x10, 0x29, 0x03, 0xD0, 0x05, 0xA9, 0x00, 0x8D, 0x01, 0x20,
           0xA9, 0x18, 0x8D, 0x01, 0x20, 0xAD, 0x16, 0x40, 0x85, 0x11, 0x68, 0x40),
    ])
    return nrom_bytes(2, code=parts, reset=0x8000, nmi=0x9000, irq=0x9000)


ROMS = {
    "wait": wait_rom,
    "random": lambda: synthrom.make_rom(5).rom,
    "nrom128": lambda: synthrom.make_rom(6, prg_banks=1).rom,
    "split": lambda: synthrom.make_rom(7, split=True).rom,
    "idle": idle_rom,
    "features": feature_rom,
    "oam": oam_rom,
    "stack_wrap": stack_wrap_rom,
    "io_corner": io_corner_rom,
    "address_wrap": address_wrap_rom,
}


def agree(rom: bytes, n: int, frameskip: int, steps: int, seed: int) -> None:
    a, lanes, b = (abi.Batch(rom, n, frameskip=frameskip) for _ in range(3))
    lanes.set_lane_kernel(True)
    sample = sorted({0, 1 % n, n // 2, n - 1, *np.random.default_rng(n).integers(0, n, 12).tolist()})
    for k in range(steps):
        m = masks_for(seed, n, k)
        for batch, stats in ((a, 0), (lanes, 0), (b, 1)):
            batch.set_actions(m)
            batch.step(auto_reset=k % 3 == 1, stats_mode=stats)
        for view in (abi.VIEW_REWARDS, abi.VIEW_DONES, abi.VIEW_RAM):
            want = b.host(view)
            assert np.array_equal(a.host(view), want), f"step {k} view {view}"
            assert np.array_equal(lanes.host(view), want), f"step {k} view {view}, lane kernel"
    assert a.step_choices()[0] >= 1 and lanes.step_choices() == (0, 0)
    # A console stopped by an illegal opcode in the middle of a step keeps the
    # step's earlier vblank only under statistics (which capture every one).
    assert np.array_equal(a.host(abi.VIEW_PRESENT), lanes.host(abi.VIEW_PRESENT))
    for e in np.flatnonzero((a.host(abi.VIEW_PRESENT) != b.host(abi.VIEW_PRESENT)).any(axis=1)):
        assert a.save_state(int(e))[O.OFF["fault"]] & 1, f"presentation record of console {e}"
    for e in sample:
        want = b.save_state(e)
        for got in (a.save_state(e), lanes.save_state(e)):
            assert np.array_equal(got, want), f"console {e}: {first_diff(got, want)}"


@pytest.mark.gpu
@pytest.mark.parametrize("name", sorted(ROMS))
@pytest.mark.parametrize("n", [60, 4160])
def test_programs_agree_with_the_lane_kernel(name, n):
    """60 consoles: the solo form; 4,160: two workgroups on some CUs."""
    say(f"[gpu] wave kernel: {name} N={n}")
    agree(ROMS[name](), n, 4, 9, 31)


@pytest.mark.gpu
@pytest.mark.parametrize("n,frameskip", [(1, 1), (2, 3), (257, 4), (700, 2), (1500, 4), (2814, 4), (4096, 1), (4097, 5),
                                         (8200, 4), (32768, 1)])
def test_sizes_agree_with_the_lane_kernel(n, frameskip):
    """1, 2, 4, 8, 12 and 16 waves per workgroup, the last one ragged (2,814
    consoles in workgroups of 12 end past the row pitch of 2,816), the ends of
    both forms' ranges."""
    say(f"[gpu] wave kernel: N={n} fs={frameskip}")
    agree(synthrom.make_rom(2026).rom, n, frameskip, 4, 77)


@pytest.mark.gpu
@pytest.mark.parametrize("n,frameskip", [(6143, 2), (6145, 1), (9205, 2), (9217, 1), (18421, 4)])
def test_workgroups_of_twelve_waves_agree_with_the_lane_kernel(n, frameskip):
    """Both sides of the sizes that take 12 waves per workgroup instead of 16,
    ragged: one, one and a half and three rounds of workgroups on the chip."""
    say(f"[gpu] wave kernel, 12 or 16 waves: N={n} fs={frameskip}")
    agree(synthrom.make_rom(2026).rom, n, frameskip, 4, 78)


def poll_rom() -> bytes:
    """Reads of $2007 and $4015 and PRG RAM traffic without end: nearly every
    instruction takes the general path."""
    loop = [0xAD, 0x07, 0x20, 0x8D, 0x00, 0x60, 0xEE, 0x00, 0x60, 0xAD, 0x15, 0x40, 0x4C, 0x00, 0x80]
    return nrom_bytes(2, code={0x8000: loop, 0x9000: [0x40]}, reset=0x8000, nmi=0x9000, irq=0x9000)


def polled(b: abi.Batch, run, steps: int, pads: np.ndarray) -> None:
    """`steps` frame-skip-1 steps of poll_rom through `run`, all enqueued
    before any is waited for; sampled consoles end as the oracle's."""
    rom = poll_rom()
    sample = (0, b.n // 2, b.n - 1)
    for _ in range(steps):
        run()
    for e in sample:
        c = O.Oracle(rom)
        c.set_reward()
        for _ in range(steps):
            c.step(int(pads[e]), 1)
        got, want = b.save_state(e), c.save()
        assert np.array_equal(got, want), f"console {e}: {first_diff(got, want)}"


@pytest.mark.gpu
@pytest.mark.parametrize("n", [60, 8200])
def test_polling_program_moves_to_the_lane_kernel(n):
    """The first step runs with one console per wave and reports; the lane
    kernel takes the next 64, then one is tried again.  Nothing here waits
    between the steps."""
    say(f"[gpu] kernel choice: polling program N={n}")
    b, pads = abi.Batch(poll_rom(), n, frameskip=1), masks_for(8, n, 0)
    b.set_actions(pads)
    polled(b, b.step, 70, pads)
    assert b.step_choices() == (2, 68)


def waiting_rom(work: int, reads: int) -> bytes:
    """An NMI handler of `work` turns of a loop and `reads` reads of $4015; the
    main program waits in JMP *."""
    turn = [0xB5, 0x10, 0x18, 0x75, 0x11, 0x95, 0x12, 0x0A, 0x2A, 0x65, 0x13, 0xCA]
    read = [0xAD, 0x15, 0x40, 0x88]
    nmi = [0xA2, work, *turn, 0xD0, 0x100 - len(turn) - 2, 0xA0, reads, *read, 0xD0, 0x100 - len(read) - 2, 0xE6, 0x20, 0x40]
    reset = [0x78, 0xA2, 0xFF, 0x9A, 0xA9, 0x80, 0x8D, 0x00, 0x20, 0x4C, 0x09, 0x80]
    return nrom_bytes(2, code={0x8000: reset, 0x9000: nmi}, reset=0x8000, nmi=0x9000, irq=0x9000)


@pytest.mark.gpu
@pytest.mark.parametrize("work,reads,stays", [(4, 5, True), (4, 100, False), (200, 100, True)])
def test_waiting_programs_are_judged_by_their_share_of_a_frame(work, reads, stays):
    """4,100 consoles (us per step of four frames, one console per wave against
    lanes): 5 reads beside a long wait, 100 beside it (about 1,300 and 800),
    100 beside 5,200 cycles of work (1,750 and 3,700)."""
    n = 4100
    say(f"[gpu] kernel choice: waiting program work={work} reads={reads} N={n}")
    b = abi.Batch(waiting_rom(work, reads), n, frameskip=4)
    b.set_actions(masks_for(8, n, 0))
    b.set_lane_kernel(True)        # past power-on
    for _ in range(2):
        b.step()
    b.set_lane_kernel(False)
    for _ in range(2):
        b.step()
    assert b.step_choices() == ((2, 0) if stays else (1, 1))


@pytest.mark.gpu
def test_captured_steps_choose_when_they_run():
    """A step captured before any has run: the replays of its graph move to the
    lane kernel as eager steps do, and the eager steps between them count."""
    import torch

    n = 60
    say(f"[gpu] kernel choice: captured step N={n}")
    b, pads = abi.Batch(poll_rom(), n, frameskip=1), masks_for(8, n, 0)
    stream = torch.cuda.Stream()
    b.set_stream(stream.cuda_stream)
    b.set_actions(pads)
    b.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        b.step()
    assert b.step_choices() == (0, 0)
    turn = iter(range(1000))

    def run():
        if next(turn) % 3 == 2:
            b.step()
        else:
            with torch.cuda.stream(stream):
                graph.replay()

    polled(b, run, 70, pads)
    assert b.step_choices() == (2, 68)


@pytest.mark.gpu
@pytest.mark.parametrize("n,chooses", [(60, True), (4097, True), (32768, True), (32769, False)])
def test_ordinary_programs_stay_with_one_console_per_wave(n, chooses):
    """Above 32,768 consoles, and under statistics, there is no choice."""
    say(f"[gpu] kernel choice: ordinary program N={n}")
    b = abi.Batch(synthrom.make_rom(5).rom, n, frameskip=2)
    for k in range(5):
        b.set_actions(masks_for(9, n, k))
        b.step(stats_mode=1 if k == 2 else 0)
    assert b.step_choices() == ((4, 0) if chooses else (0, 0))


@pytest.mark.gpu
@pytest.mark.parametrize("value,chooses", [("8", False), ("16", False), ("5", True), ("", True)])
def test_waves_per_group_asks_for_the_lane_kernel(value, chooses):
    """NESLE_WAVES_PER_GROUP shapes the lane kernel's workgroups, so with a
    value it takes (4, 8 or 16) that kernel runs; read once per process."""
    say(f"[gpu] NESLE_WAVES_PER_GROUP={value!r}")
    code = ("from nesle_amd import abi, synthrom; import numpy as np\n"
            "b = abi.Batch(synthrom.make_rom(5).rom, 300, frameskip=1)\n"
            "b.set_actions(np.zeros(300, np.uint8)); b.step(); b.step(); print(b.step_choices())")
    out = subprocess.run([sys.executable, "-c", code], env={**os.environ, "NESLE_WAVES_PER_GROUP": value},
                         cwd=build.ROOT, capture_output=True, text=True, timeout=100)
    assert out.returncode == 0, out.stderr
    assert out.stdout.split("\n")[-2] == ("(2, 0)" if chooses else "(0, 0)"), out.stdout


def vector_rom(irq: int, flow: list[int]) -> bytes:
    """Flow at $FFF5 (padded with NOPs) into vectors whose bytes are all NOPs
    but the last; the code they point to counts and comes back."""
    back = [0xE6, 0x20, 0xA5, 0x20, 0x85, 0x00, 0x49, 0xFF, 0x85, 0x01, 0x4C, 0xF5, 0xFF]   # count; JMP $FFF5
    return nrom_bytes(2, code={0xEAEA: back, irq: back, 0xFFF5: (flow + [0xEA] * 5)[:5]}, reset=0xEAEA, nmi=0xEAEA, irq=irq)


@pytest.mark.gpu
@pytest.mark.parametrize("irq,flow", [
    (0xEAEA, []),                    # NOPs over the end: the next instruction is RAM's
    (0xADEA, []),                    # LDA abs at $FFFF: its operand is RAM $0000-$0001
    (0xA5EA, []),                    # LDA zp at $FFFF
    (0xEA8D, []),                    # STA abs at $FFFE
    (0xADEA, [0x4C, 0xFF, 0xFF]),    # the same instruction entered by a jump
    (0xEAEA, [0x18, 0x90, 0x06]),    # a branch over the end
    (0x9090, [0x18, 0x90, 0x02]),    # a branch to the vectors
    # Three bytes at $FFF7 fall into $FFFA, past operands that are no opcodes.
    (0xADEA, [0xEA, 0xEA, 0xAD, 0x02, 0x03]),
    (0xADEA, [0xEA, 0xEA, 0x8D, 0x02, 0x03]),
    (0xEA8D, [0xEA, 0xEA, 0xAD, 0x02, 0x03]),
])
def test_flow_over_the_vectors_matches_oracle(irq, flow):
    rom = vector_rom(irq, flow)
    b, cons = abi.Batch(rom, 3, frameskip=2), [O.Oracle(rom) for _ in range(3)]
    for c in cons:
        c.set_reward()
    stopped = set()
    for k in range(4):
        m = masks_for(3, 3, k)
        b.set_actions(m)
        b.step()
        for e, c in enumerate(cons):
            if e in stopped:
                continue
            try:
                c.step(int(m[e]), 2)
            except RuntimeError:       # an illegal opcode: the oracle's PC has moved past it
                stopped.add(e)
                assert b.save_state(e)[O.OFF["fault"]] & 1
                continue
            got, want = b.save_state(e), c.save()
            assert np.array_equal(got, want), f"step {k} console {e}: {first_diff(got, want)}"


HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not Path(HIPCC).exists(), reason="hipcc not available")
@pytest.mark.parametrize("source", ["nes_step_wave.hip", "nes_step_solo.hip"])
def test_two_workgroups_share_a_cu(tmp_path, source):
    """Eight waves per SIMD: at most 80 KB of LDS, 80 scalar registers (800
    per SIMD in units of 16) and 64 vector registers, and no scratch."""
    out = tmp_path / "wave.s"
    path = build.CSRC / source
    subprocess.run([HIPCC, "--offload-arch=gfx950", "--offload-device-only", "-S", *build.source_flags(path), "-o",
                    str(out), str(path)], check=True, capture_output=True, text=True)
    meta = out.read_text().split("amdhsa.kernels:", 1)[1]
    value = {k: int(v) for k, v in re.findall(r"\.(group_segment_fixed_size|private_segment_fixed_size|sgpr_count|"
                                              r"vgpr_count):\s+(\d+)", meta)}
    assert value["group_segment_fixed_size"] <= 80 * 1024 and value["private_segment_fixed_size"] == 0
    assert value["sgpr_count"] <= 80 and value["vgpr_count"] <= 64
