// nes_choice.h -- which kernel steps a batch: plain rules shared by the host
// library and the step kernels, compiled alone by the CPU tests.
#pragma once

#include <cstddef>
#include <cstdint>

#include "nes_micro.h"

#ifdef __HIPCC__
#define NESLE_BOTH_SIDES __host__ __device__
#else
#define NESLE_BOTH_SIDES
#endif

namespace nesle {

// Whether straight-line flow into the vectors ($FFFA-$FFFF) meets no
// instruction whose bytes run past $FFFF (they would wrap to RAM), which the
// assembly of the one-console-per-wave kernels (nes_wave.h) would read from
// its guard bytes.  Those kernels enter an instruction anywhere below $FFFA by
// a jump or a branch, so every start there counts; from $FFFA on what falls
// into what is given by the image.  (Jumps to the vectors are not flow in this
// sense: the kernels run those instructions one at a time.)  Starts below
// $FFF0 add nothing: what they fall into is a start itself.
inline bool closed_end(const std::uint8_t* prg, std::size_t size) {
    constexpr std::uint32_t kTail = 16, kVectors = kTail - 6;
    bool reached[kTail] = {};
    for (std::uint32_t o = 0; o < kVectors; ++o) reached[o] = true;
    for (std::uint32_t o = 0; o < kTail; ++o) {
        if (!reached[o]) continue;
        const auto& w = mc::kTableFull.e[prg[size - kTail + o]];
        if (w.d[14] & mc::kIllegal) continue;
        const std::uint32_t next = o + ((w.d[0] >> 12) & 3);
        if (next > kTail) return false;
        // JMP, JSR, RTS, RTI and BRK do not go on to the next instruction.
        const bool leaves = w.d[9] != 0 || w.d[10] != 0 || w.d[11] != 0 || (w.d[14] & mc::kJmpInd) != 0;
        if (!leaves && next < kTail) reached[next] = true;
    }
    return true;
}

// The choice between the one-console-per-wave kernels and the lane kernel, in
// device memory.  A program the first gain on seldom leaves their assembly
// for the general path (NMI entry, DMA, PPU control: about a dozen times a
// frame); one that runs from RAM or polls other registers all the time goes to
// the lane kernel for a while and is then tried again, for one step at first: a
// step wholly on the general path takes some 430 ms at 32,768 consoles, against
// the lane kernel's 17, so the while grows from 64 steps by fours to 4,096
// (0.6 % of them) and is 64 again once a run of steps as long as it went well.
//
// A step launches both kernels and the one that is not chosen returns at once:
// the per-wave kernel reads `next` and leaves it in `now` for the lane kernel
// behind it, which counts the step (choice_update).  So each step's choice
// follows from the steps before it on the stream, whether they were enqueued
// long before any of them ran or are replayed from a captured graph.  Only the
// kernel depends on it, not the results.  The launch that returns at once costs
// 3 us of the vector environment's 711 with one console, 9 of 3,517 at 30,001
// consoles.
constexpr std::uint32_t kGeneralSlots = 16;
struct StepChoice {
    std::uint64_t steps[2];             // taken by [0] one console per wave, [1] the lane kernel
    std::uint32_t next, now;            // kernel of the next step, of this one
    std::uint32_t left;                 // steps the lane kernel still takes
    std::uint32_t level, good;          // its next stay, kLaneSteps << 2 level; good steps since the last one
    std::uint32_t over[kGeneralSlots];  // whether the first consoles took the general path too often
};
constexpr std::uint32_t kLaneSteps = 64, kMaxLevel = 3;

// After the step whose kernel is `now`: the next one's.
NESLE_BOTH_SIDES inline void choice_update(StepChoice& c) {
    ++c.steps[c.now];
    if (c.now == 0) {
        std::uint32_t over = 0;
        for (std::uint32_t i = 0; i < kGeneralSlots; ++i) over |= c.over[i];
        const std::uint32_t stay = kLaneSteps << 2 * c.level;
        if (over == 0) {
            if (c.level != 0 && ++c.good >= stay) c.level = c.good = 0;
            return;
        }
        c.next = 1;
        c.left = stay;
        c.good = 0;
        if (c.level < kMaxLevel) ++c.level;
    } else if (--c.left == 0) {
        c.next = 0;
    }
}

// Trips through the general path per frame from which on the lane kernel is
// quicker on a batch of n consoles: `idle` of them, and `busy` more for a frame
// that never waits in a jump to itself.  Both kernels skip those jumps, so a
// program that waits for its NMI costs the lane kernel as little as its share
// of a busy frame says, and fewer trips outweigh it.  In ms per step of four
// frames, with w waves of one console per SIMD (1,024 consoles each), measured
// on programs of 0 to 500 reads of $4015 a frame beside 60 to 2,600 other
// instructions and a wait: the lane kernel 0.12 and, for a busy frame of 3.5
// cycles an instruction, 15 up to 8,192 consoles or 18; one console per wave
// 0.05 and 0.39 w, at least 2.4; a trip 1,660 cycles of 2.4 GHz per wave, of at
// least 2.4 waves.  At 4,096 consoles 6 + 1,139 trips, 8,192 3 + 537, 16,384
// 2 + 265, 32,768 1 + 62.
struct GeneralLimit {
    float idle, busy;
};
inline GeneralLimit general_limit(std::uint32_t n) {
    const double w = n / 1024.0;
    const double trip_ms = 4 * 1660.0 * (w > 2.4 ? w : 2.4) / 2.4e6;
    const double lane_ms = n <= 8192 ? 15.0 : 18.0, wave_ms = 0.39 * w > 2.4 ? 0.39 * w : 2.4;
    return {static_cast<float>((0.12 - 0.05) / trip_ms), static_cast<float>((lane_ms - wave_ms) / trip_ms)};
}

// Whether a console's step of `frames` frames, with `trips` trips and `jumps`
// skipped jumps (9 dots each) of the frames' `dots`, is over it.
NESLE_BOTH_SIDES inline bool over_limit(GeneralLimit l, std::uint32_t trips, std::uint32_t jumps, std::uint32_t frames,
                                        std::uint32_t dots) {
    const float n = static_cast<float>(frames), waits = 9.0f * static_cast<float>(jumps) / static_cast<float>(dots);
    return static_cast<float>(trips) > l.idle * n + l.busy * (waits < n ? n - waits : 0.0f);
}

}  // namespace nesle
