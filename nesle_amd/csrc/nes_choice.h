// nes_choice.h -- which kernel steps a batch: rules without device code of
// their own, shared by the host library and compiled alone by the CPU tests.
#pragma once

#include <cstddef>
#include <cstdint>

#include "nes_micro.h"

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

}  // namespace nesle
