// nes_wave.h -- the 6502 of the one-console-per-wave step kernels
// (nes_step_wave.hip): the instructions a console spends nearly all its time
// in, as threaded code on the scalar unit.
//
// A wave that serves one console has no use for 64 copies of a datapath:
// registers, flags and time live in scalar registers, every opcode is its own
// few instructions and the next opcode's code is entered by a computed jump.
// The compiler offers no computed jump on this target (a switch becomes a
// tree of compares, about 16 instructions deep for 256 opcodes, and an
// `asm goto` an exit chain through all its labels), hence assembly.  The
// block runs instructions from PRG ROM whose operands lie in RAM, PRG ROM, the
// I/O registers programs poll ($2002, $2004, $4016) or those they write in
// numbers ($2000, $2001, $2005, $2006, $2007 to the nametables, $4000-$4016
// but $4014), and leaves with
//   kWaveEvent    an instruction reached the next PPU event; it is complete;
//   kWaveStore    the instruction stores `value` at `addr`, another register
//                 or PRG RAM: all of it but the store is done, its time
//                 included (which may have reached the event);
//   kWaveGeneral  the next instruction is for the general path (other I/O
//                 reads, PRG RAM, illegal opcodes, JMP indirect, stack and
//                 zero-page pointer wraps, loops that wait -- a jump to
//                 itself, a branch back to its read of $2002 --, a target
//                 outside PRG ROM or among the vectors): nothing of it has
//                 run.
//
// Registers.  The countdown holds the dots to the next event less one, so
// that subtracting an instruction's dots borrows exactly when it reaches the
// event.  N and Z stay as the last result: Z is set when bits 0-7 of NZ are
// zero, N when bit 7 or bit 15 is set (BIT and pulled flags, whose N and Z do
// not come from one byte, use bit 15).  V is bit 7 of V1 & V2.  W is the
// instruction shifted left by eight: opcode in bits 8-15, operand bytes in
// bits 16-31 (vT holds it too, for the vector unit).  The PC is an LDS
// address in vF.  No instruction checks whether its successor lies past the
// PRG image: the host runs only images here whose straight-line flow cannot
// get there in the middle of an instruction (closed_end, nes_choice.h), 128
// bytes of an illegal opcode stand on either side of the image (a branch
// leaves it downwards by at most that), and jumps test their target.
//
// Dispatch.  Each opcode's code starts at table + 256 * opcode; the table is
// 64 KB long and 64 KB aligned, so a jump's target is the table's address
// with W's low half in place of its own: two scalar instructions.  While an
// instruction runs, the window of eight bytes at the next one is already
// read, and its opcode and operands picked from it (v_perm); the read issued
// is the window after that, so no instruction waits for its own bytes except
// after a jump.  LDS: PRG ROM at kWaveRom, this console's 2 KB of RAM,
// aligned to their size, at `ram`.  Only lane 0 is active inside: the reads
// are unaligned, and an unaligned LDS read takes four cycles per active lane.
//
// Two forms (the symbol SOLO), by what bounds a wave.  Measured per SIMD: a
// scalar instruction 4.3 cycles of issue, a vector one as much on a pipe of
// its own, a branch not taken about 1 but 13 of the wave's own time, a branch
// on vcc 29, v_readfirstlane to a scalar use 21, s_setpc 32, an LDS read 64.
//   SOLO = 1, few waves per SIMD (the wave's own time bounds): an event
//   selects another table, all of whose entries leave the block, instead of
//   branching, in the shadow of the operand's read.
//   SOLO = 0, many waves (both units bound, at 6.1 scalar and 6.3 vector
//   instructions per emulated one, 30 cycles per SIMD): the countdown is a
//   vector register and the event a branch on its borrow.
// At 1,000 consoles the first takes 2.47 ms per 4-frame step, the second
// 2.80; at 8,192 3.92 and 3.43.  A store that leaves the block costs 200
// scalar instructions and the way back in; done inside, a program that fills
// nametables in a loop takes 4.0 ms instead of 12.1 (64 consoles), 27 instead
// of 141 (32,768).
//
// Addresses are formed on the vector unit (SDWA picks the operand byte out of
// vT), and read-modify-write results are too.
//
// Hazards.  Assembly text gets no wait states from the compiler.  A scalar
// register written by v_readfirstlane is read by scalar instructions, or by a
// vector one at least two instructions later; a vector register written by a
// vector instruction is read by v_readfirstlane at least one instruction
// later, and likewise after a partial (dst_sel) SDWA write; every LDS read is
// waited for before the first use of its result and before the block ends.
#pragma once

#include <cstdint>

namespace nesle {

constexpr std::uint32_t kWaveRom = 256;
constexpr std::uint32_t kWaveRomEnd = 0x7FFA;   // offsets from here on: the vectors
constexpr std::uint32_t kWaveGuard = 128;       // bytes of an illegal opcode on either side of the image
// The console's register area (reg::, nes_step.hip) as the block reads it: v at
// 16 and t at 18, fine x at 6, the scrolls at 8 and 9, ctrl at 0, and after
// those 40 bytes
constexpr std::uint32_t kWaveVram = 40;    // address of the nametables (64 bits)
constexpr std::uint32_t kWaveApu = 48;     // address of the $4000 byte (64 bits)
constexpr std::uint32_t kWavePitch = 56;   // of the rows from there
constexpr std::uint32_t kWaveNt = 60;      // mirroring: offset = (i & low half) | (i >> 1 & high half)
constexpr std::uint32_t kWaveRegsBytes = 64;
enum : std::uint32_t { kWaveGeneral = 0, kWaveEvent = 1, kWaveStore = 2 };

struct WaveCpu {
    std::uint32_t pc;                 // 16-bit address, $8000-$FFFD on entry
    std::uint32_t a, x, y, sp, p;
    std::uint32_t io, flags;          // the kernel's packed I/O registers
    std::int32_t left;                // dots to the next PPU event, positive on entry
    std::uint32_t addr, value;        // of a kWaveStore
};

// Runs until one of the conditions above.  `brk`: the BRK vector.
__device__ __forceinline__ std::uint32_t wave_run(WaveCpu& c, std::uint32_t ram, std::uint32_t regs, std::uint32_t brk) {
    std::uint32_t pc = c.pc - 0x8000u + kWaveRom, left = static_cast<std::uint32_t>(c.left - 1);
    std::uint32_t a = c.a, x = c.x, y = c.y, sp = c.sp, p = c.p, io = c.io, fl = c.flags, why, addr, value;
    // The vector's LDS address; 0: not an address the block runs from.
    const std::uint32_t vec = brk - 0x8000u < kWaveRomEnd ? brk - 0x8000u + kWaveRom : 0u;
    asm volatile(".set SOLO, " NESLE_WAVE_SOLO R"(
; ---- registers ------------------------------------------------------------
.set rLim, 34
.set rA, 35
.set rX, 36
.set rY, 37
.set rSP, 38
.set rP, 39
.set rNZ, 40
.set rC, 41
.set rV1, 42
.set rV2, 43
.set rL, 44
.set rW, 45
.set rT, 46
.set rU, 47
.set rR, 48
.set rM, 49
.set rFF, 50
.set r2G, 51
.set r2000, 52
.set rLo, 53
.set rIO, 54
.set rFL, 55
.set rJ, 56
.set rRet, 58
.set rTab, 60
.set rK, 61
.set rCall, 62
.set rVec, 64
.set rSel0, 65
.set rSel1, 66
.set rSel2, 67
.set rSel3, 68
.set rExit, 69
.set rQ, 70
.set vW, 8
.set vF, 10
.set vA, 11
.set vM, 12
.set vD, 13
.set vRAM, 15
.set v7FF, 16
.set vT, 17
.set vL, 18
.set vRG, 19
.set vZ, 20
.set vP, 22
.set ROM, 256
.set LIM, 256 + 0x7FF9

; ---- fetch, time and dispatch ------------------------------------------------
; The next instruction's bytes are in the window already read, \len bytes on;
; the window of eight bytes at the next instruction is read for the one after
; it.  \k LDS operations have been issued since the handler began.  W is the
; next instruction's from here on.
.macro AHEAD len, k=0
  s_waitcnt lgkmcnt(\k)
  v_perm_b32 v[vT], v[vW+1], v[vW], s[rSel\len]
  v_add_u32 v[vF], \len, v[vF]
  ds_read_b64 v[vW:vW+1], v[vF]
  v_readfirstlane_b32 s[rW], v[vT]
.endm
; AIM forms the jump's target, GO jumps.
.macro AIM
.if SOLO
  s_pack_lh_b32_b16 s[rJ], s[rW], s[rQ]
.else
  s_pack_lh_b32_b16 s[rJ], s[rW], s[rTab]
.endif
.endm
.macro GO
  s_setpc_b64 s[rJ:rJ+1]
.endm
; After a jump: its window has been read at \at.
.macro ENTER at, off=0
  ds_read_b64 v[vW:vW+1], v[\at] offset:\off
.endm
.macro ENTERED
  s_waitcnt lgkmcnt(0)
  v_perm_b32 v[vT], v[vW+1], v[vW], s[rSel0]
  s_nop 0
  v_readfirstlane_b32 s[rW], v[vT]
  AIM
  GO
.endm
.macro TIME dots
.if SOLO
  s_sub_u32 s[rL], s[rL], \dots
.else
  v_subrev_co_u32 v[vL], vcc, \dots, v[vL]
.endif
.endm
; Time of an instruction, the PC being at the next one.
.macro PASS dots, event
  TIME \dots
.if SOLO
  s_cselect_b32 s[rQ], s[rExit], s[rTab]
.else
  s_cbranch_vccnz \event
.endif
.endm
.macro NEXT dots
  PASS \dots, .Lw%=_exit
  AIM
  GO
.endm
; Finishes an instruction that leaves the block in the middle of its read.
.macro DONE n, op:vararg
.if SOLO == 0
  .subsection 1
.Lw%=_event\n:
  s_waitcnt lgkmcnt(0)
  \op
  s_branch .Lw%=_exit
  .subsection 0
.endif
.endm
; rR: bit 8 set when indexing crossed a page (one cycle more).
.macro CROSS dots
  s_bitcmp1_b32 s[rR], 8
  s_cselect_b32 s[rR], \dots+3, \dots
.endm

; ---- operands ------------------------------------------------------------------
.macro ZP
  v_or_b32_sdwa v[vA], v[vRAM], v[vT] dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:DWORD src1_sel:BYTE_2
.endm
.macro ZPI i
  v_add_u32_sdwa v[vA], s[\i], v[vT] dst_sel:BYTE_0 dst_unused:UNUSED_PAD src0_sel:DWORD src1_sel:BYTE_2
  s_nop 0
  v_or_b32 v[vA], v[vRAM], v[vA]
.endm
.macro ABS other
  s_cmp_ge_u32 s[rW], s[r2G]
  s_cbranch_scc1 \other
  v_bfe_u32 v[vA], v[vT], 16, 11
  v_or_b32 v[vA], v[vRAM], v[vA]
.endm
; The address in rT.
.macro AT other
  s_cmp_ge_u32 s[rT], s[r2000]
  s_cbranch_scc1 \other
  v_and_or_b32 v[vA], s[rT], v[v7FF], v[vRAM]
.endm
.macro IDX i
  s_lshr_b32 s[rU], s[rW], 16
  s_add_u32 s[rT], s[rU], s[\i]
  s_xor_b32 s[rR], s[rT], s[rU]
.endm
; The zero-page pointer at byte rT (at $FF its high byte wraps to $00, left to
; the general path) into rU.
.macro POINTER
  s_cmp_eq_u32 s[rT], s[rFF]
  s_cbranch_scc1 .Lw%=_general
  v_or_b32 v[vA], s[rT], v[vRAM]
  ds_read_u16 v[vM], v[vA]
  s_waitcnt lgkmcnt(0)
  v_readfirstlane_b32 s[rU], v[vM]
.endm
.macro PTRX
  s_bfe_u32 s[rT], s[rW], s[rLo]
  s_add_u32 s[rT], s[rT], s[rX]
  s_and_b32 s[rT], s[rT], s[rFF]
  POINTER
  s_mov_b32 s[rT], s[rU]
.endm
.macro PTRY
  s_bfe_u32 s[rT], s[rW], s[rLo]
  POINTER
  s_add_u32 s[rT], s[rU], s[rY]
  s_xor_b32 s[rR], s[rT], s[rU]
.endm
; A read at rT outside RAM: PRG ROM, or an I/O register whose byte comes back
; in rM (an indexed address past $FFFF has bit 15 clear and is left to the
; general path with the other I/O addresses).
.macro ROMIO n, len
  .subsection 1
.Lw%=_rom\n:
  s_bitcmp0_b32 s[rT], 15
  s_cbranch_scc1 .Lw%=_io\n
  s_bitset0_b32 s[rT], 15
  v_mov_b32 v[vA], s[rT]
  ds_read_u8 v[vM], v[vA] offset:256
  s_branch .Lw%=_got\n
.Lw%=_io\n:
  s_call_b64 s[rCall:rCall+1], .Lw%=_ioread
  v_mov_b32 v[vM], s[rM]
  AHEAD \len
  s_branch .Lw%=_time\n
  .subsection 0
.endm

; ---- operations on the byte in vM ------------------------------------------------
.macro BYTE
  v_readfirstlane_b32 s[rM], v[vM]
.endm
.macro OP_LD r
  v_readfirstlane_b32 s[\r], v[vM]
  v_readfirstlane_b32 s[rNZ], v[vM]
.endm
.macro OP_ORA r
  BYTE
  s_or_b32 s[rA], s[rA], s[rM]
  s_mov_b32 s[rNZ], s[rA]
.endm
.macro OP_AND r
  BYTE
  s_and_b32 s[rA], s[rA], s[rM]
  s_mov_b32 s[rNZ], s[rA]
.endm
.macro OP_EOR r
  BYTE
  s_xor_b32 s[rA], s[rA], s[rM]
  s_mov_b32 s[rNZ], s[rA]
.endm
.macro ADD
  s_add_u32 s[rNZ], s[rA], s[rM]
  s_add_u32 s[rNZ], s[rNZ], s[rC]
  s_xor_b32 s[rV1], s[rA], s[rNZ]
  s_xor_b32 s[rV2], s[rM], s[rNZ]
  s_lshr_b32 s[rC], s[rNZ], 8
  s_and_b32 s[rA], s[rNZ], s[rFF]
.endm
.macro OP_ADC r
  BYTE
  ADD
.endm
.macro OP_SBC r
  BYTE
  s_xor_b32 s[rM], s[rM], s[rFF]
  ADD
.endm
.macro OP_CP r
  BYTE
  s_sub_u32 s[rM], s[\r], s[rM]
  s_cselect_b32 s[rC], 0, 1
  s_and_b32 s[rNZ], s[rM], s[rFF]
.endm
.macro OP_BIT r
  BYTE
  s_lshl_b32 s[rV1], s[rM], 1
  s_movk_i32 s[rV2], 0x80
  s_lshr_b32 s[rT], s[rM], 7
  s_lshl_b32 s[rT], s[rT], 15
  s_and_b32 s[rNZ], s[rA], s[rM]
  s_or_b32 s[rNZ], s[rNZ], s[rT]
.endm
; Read-modify-write: the result in vD (its low byte is written) and rNZ.
.macro MOP_INC
  v_add_u32 v[vD], 1, v[vM]
  ds_write_b8 v[vA], v[vD]
  v_readfirstlane_b32 s[rNZ], v[vD]
.endm
.macro MOP_DEC
  v_subrev_u32 v[vD], 1, v[vM]
  ds_write_b8 v[vA], v[vD]
  v_readfirstlane_b32 s[rNZ], v[vD]
.endm
.macro MOP_ASL
  v_lshlrev_b32 v[vD], 1, v[vM]
  ds_write_b8 v[vA], v[vD]
  v_readfirstlane_b32 s[rNZ], v[vD]
  s_lshr_b32 s[rC], s[rNZ], 8
.endm
.macro MOP_ROL
  v_lshl_or_b32 v[vD], v[vM], 1, s[rC]
  ds_write_b8 v[vA], v[vD]
  v_readfirstlane_b32 s[rNZ], v[vD]
  s_lshr_b32 s[rC], s[rNZ], 8
.endm
.macro MOP_LSR
  v_lshrrev_b32 v[vD], 1, v[vM]
  v_readfirstlane_b32 s[rM], v[vM]
  ds_write_b8 v[vA], v[vD]
  v_readfirstlane_b32 s[rNZ], v[vD]
  s_and_b32 s[rC], s[rM], 1
.endm
.macro MOP_ROR
  s_lshl_b32 s[rT], s[rC], 8
  v_or_b32 v[vD], s[rT], v[vM]
  v_readfirstlane_b32 s[rM], v[vM]
  v_lshrrev_b32 v[vD], 1, v[vD]
  ds_write_b8 v[vA], v[vD]
  v_readfirstlane_b32 s[rNZ], v[vD]
  s_and_b32 s[rC], s[rM], 1
.endm
; One register in place.
.macro ROP_ASL r
  s_lshl_b32 s[rNZ], s[\r], 1
  s_lshr_b32 s[rC], s[rNZ], 8
  s_and_b32 s[\r], s[rNZ], s[rFF]
.endm
.macro ROP_ROL r
  s_lshl1_add_u32 s[rNZ], s[\r], s[rC]
  s_lshr_b32 s[rC], s[rNZ], 8
  s_and_b32 s[\r], s[rNZ], s[rFF]
.endm
.macro ROP_LSR r
  s_and_b32 s[rC], s[\r], 1
  s_lshr_b32 s[\r], s[\r], 1
  s_mov_b32 s[rNZ], s[\r]
.endm
.macro ROP_ROR r
  s_lshl_b32 s[rT], s[rC], 8
  s_or_b32 s[rT], s[rT], s[\r]
  s_and_b32 s[rC], s[\r], 1
  s_lshr_b32 s[\r], s[rT], 1
  s_mov_b32 s[rNZ], s[\r]
.endm
.macro ROP_INC r
  s_add_u32 s[rNZ], s[\r], 1
  s_and_b32 s[\r], s[rNZ], s[rFF]
.endm
.macro ROP_DEC r
  s_sub_u32 s[rNZ], s[\r], 1
  s_and_b32 s[\r], s[rNZ], s[rFF]
.endm

; ---- opcode code, in opcode order ------------------------------------------------
.macro H
  .p2align 8
.endm
.macro ILL n=1
  .rept \n
  .p2align 8
  s_branch .Lw%=_general
  .endr
.endm
; Reads.
.macro LD_IMM r
  H
  s_bfe_u32 s[\r], s[rW], s[rLo]
  AHEAD 2
  s_mov_b32 s[rNZ], s[\r]
  NEXT 6
.endm
.macro R_IMM op, r
  H
  s_bfe_u32 s[rM], s[rW], s[rLo]
  AHEAD 2
  IMM_\op \r
  NEXT 6
.endm
.macro IMM_ORA r
  s_or_b32 s[rA], s[rA], s[rM]
  s_mov_b32 s[rNZ], s[rA]
.endm
.macro IMM_AND r
  s_and_b32 s[rA], s[rA], s[rM]
  s_mov_b32 s[rNZ], s[rA]
.endm
.macro IMM_EOR r
  s_xor_b32 s[rA], s[rA], s[rM]
  s_mov_b32 s[rNZ], s[rA]
.endm
.macro IMM_ADC r
  ADD
.endm
.macro IMM_SBC r
  s_xor_b32 s[rM], s[rM], s[rFF]
  ADD
.endm
.macro IMM_CP r
  s_sub_u32 s[rM], s[\r], s[rM]
  s_cselect_b32 s[rC], 0, 1
  s_and_b32 s[rNZ], s[rM], s[rFF]
.endm
; A read from \n's address in vA and what follows.
.macro READ n, len, dots, op:vararg
  ds_read_u8 v[vM], v[vA]
.Lw%=_got\n:
  AHEAD \len, 1
.Lw%=_time\n:
  PASS \dots, .Lw%=_event\n
  AIM
  s_waitcnt lgkmcnt(1)
  \op
  GO
  DONE \n, \op
.endm
.macro R_ZP op, r
  H
  ZP
  READ \@, 2, 9, OP_\op \r
.endm
.macro R_ZPI op, r, i
  H
  ZPI \i
  READ \@, 2, 12, OP_\op \r
.endm
.macro R_ABS op, r
  H
  ABS .Lw%=_abs\@
  READ \@, 3, 12, OP_\op \r
  .subsection 1
.Lw%=_abs\@:
  s_lshr_b32 s[rT], s[rW], 16
  ROMIO \@, 3
.endm
.macro R_ABSI op, r, i
  H
  IDX \i
  CROSS 12
  AT .Lw%=_rom\@
  READ \@, 3, s[rR], OP_\op \r
  ROMIO \@, 3
.endm
.macro R_INDX op, r
  H
  PTRX
  AT .Lw%=_rom\@
  READ \@, 2, 18, OP_\op \r
  ROMIO \@, 2
.endm
.macro R_INDY op, r
  H
  PTRY
  CROSS 15
  AT .Lw%=_rom\@
  READ \@, 2, s[rR], OP_\op \r
  ROMIO \@, 2
.endm
; Stores.  A store outside RAM leaves the block with the instruction otherwise
; done.
.macro STORE r
  v_mov_b32 v[vD], s[\r]
  ds_write_b8 v[vA], v[vD]
.endm
.macro OUT n, r, len, dots
  .subsection 1
.Lw%=_out\n:
  s_mov_b32 s[rM], s[\r]
  AHEAD \len
  TIME \dots
.if SOLO
  s_cselect_b32 s[rQ], s[rExit], s[rTab]
.endif
  s_branch .Lw%=_store
  .subsection 0
.endm
.macro W_ZP r
  H
  ZP
  STORE \r
  AHEAD 2, 1
  NEXT 9
.endm
.macro W_ZPI r, i
  H
  ZPI \i
  STORE \r
  AHEAD 2, 1
  NEXT 12
.endm
.macro W_ABS r
  H
  ABS .Lw%=_abs\@
  STORE \r
  AHEAD 3, 1
  NEXT 12
  .subsection 1
.Lw%=_abs\@:
  s_lshr_b32 s[rT], s[rW], 16
  OUT \@, \r, 3, 12
.endm
.macro W_ABSI r, i
  H
  s_lshr_b32 s[rT], s[rW], 16
  s_add_u32 s[rT], s[rT], s[\i]
  AT .Lw%=_out\@
  STORE \r
  AHEAD 3, 1
  NEXT 15
  OUT \@, \r, 3, 15
.endm
.macro W_INDX r
  H
  PTRX
  AT .Lw%=_out\@
  STORE \r
  AHEAD 2, 1
  NEXT 18
  OUT \@, \r, 2, 18
.endm
.macro W_INDY r
  H
  PTRY
  AT .Lw%=_out\@
  STORE \r
  AHEAD 2, 1
  NEXT 18
  OUT \@, \r, 2, 18
.endm
; Read-modify-write.
.macro M_ZP op
  H
  ZP
  READ \@, 2, 15, MOP_\op
.endm
.macro M_ZPX op
  H
  ZPI rX
  READ \@, 2, 18, MOP_\op
.endm
.macro M_ABS op
  H
  ABS .Lw%=_general
  READ \@, 3, 18, MOP_\op
.endm
.macro M_ABSX op
  H
  s_lshr_b32 s[rT], s[rW], 16
  s_add_u32 s[rT], s[rT], s[rX]
  AT .Lw%=_general
  READ \@, 3, 21, MOP_\op
.endm
.macro A_ op, r
  H
  AHEAD 1
  ROP_\op \r
  NEXT 6
.endm
; Transfer \d <- \s with flags.
.macro T_ d, s
  H
  AHEAD 1
  s_mov_b32 s[\d], s[\s]
  s_mov_b32 s[rNZ], s[\s]
  NEXT 6
.endm
; One scalar instruction.
.macro F_ insn:vararg
  H
  AHEAD 1
  \insn
  NEXT 6
.endm
; Branch: the condition sets SCC; taken when SCC is \want.
.macro BRANCH want, test:vararg
  H
  BRANCH_ \want, \test
.endm
.macro BRANCH_ want, test:vararg
  \test
  s_cbranch_scc\want .Lw%=_taken\@
  AHEAD 2
  NEXT 6
.Lw%=_taken\@:
  v_add_u32 v[vD], 2, v[vF]           ; the address after the branch
  v_add_u32_sdwa v[vF], v[vD], sext(v[vT]) dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:DWORD src1_sel:BYTE_2
  ENTER vF
  v_readfirstlane_b32 s[rU], v[vD]
  v_readfirstlane_b32 s[rT], v[vF]
  s_cmp_gt_u32 s[rT], s[rLim]
  s_cbranch_scc1 .Lw%=_back
  s_xor_b32 s[rU], s[rU], s[rT]
  s_lshr_b32 s[rU], s[rU], 8          ; SCC: another page
  s_cselect_b32 s[rU], 12, 9
  PASS s[rU], .Lw%=_exit
  ENTERED
.endm
.macro BRANCHV want
  H
  s_and_b32 s[rT], s[rV1], s[rV2]
  BRANCH_ \want, s_bitcmp1_b32 s[rT], 7
.endm
; A jump to the LDS address in rU, whose window has been read; \dots charged.
.macro JUMP dots
  v_mov_b32 v[vF], s[rU]
  PASS \dots, .Lw%=_exit
  ENTERED
.endm
; The window at the 16-bit address in \at, wherever that is; its LDS address
; into rU from the scalar copy in rT.  Outside $8000-$FFF9 to the general path.
.macro TARGET at, lo=0
  v_bfe_u32 v[vD], v[\at], \lo, 15
  ENTER vD, ROM
  s_sub_u32 s[rU], s[rT], 0x8000 - ROM
  s_sub_u32 s[rT], s[rT], 0x8000
  s_cmp_gt_u32 s[rT], LIM - ROM
  s_cbranch_scc1 .Lw%=_general
.endm
; \add more than this instruction's address into \r.
.macro HERE r, add
  v_readfirstlane_b32 s[\r], v[vF]
  s_add_u32 s[\r], s[\r], 0x8000 - ROM + \add
.endm
; P from rNZ, rC, rV1, rV2 and rP into rT.
.macro PACK
  s_and_b32 s[rT], s[rP], 0x3C
  s_or_b32 s[rT], s[rT], s[rC]
  s_and_b32 s[rU], s[rV1], s[rV2]
  s_and_b32 s[rU], s[rU], 0x80
  s_cselect_b32 s[rU], 64, 0
  s_or_b32 s[rT], s[rT], s[rU]
  s_and_b32 s[rU], s[rNZ], 0x8080
  s_cselect_b32 s[rU], 0x80, 0
  s_or_b32 s[rT], s[rT], s[rU]
  s_and_b32 s[rU], s[rNZ], s[rFF]
  s_cselect_b32 s[rU], 0, 2
  s_or_b32 s[rT], s[rT], s[rU]
  s_or_b32 s[rT], s[rT], 32
.endm
; rNZ, rC, rV1, rV2 from the P byte in rP.
.macro UNPACK
  s_and_b32 s[rC], s[rP], 1
  s_lshl_b32 s[rV1], s[rP], 1
  s_movk_i32 s[rV2], 0x80
  s_bfe_u32 s[rT], s[rP], 0x10007
  s_lshl_b32 s[rNZ], s[rT], 15
  s_bfe_u32 s[rT], s[rP], 0x10001
  s_xor_b32 s[rT], s[rT], 1
  s_or_b32 s[rNZ], s[rNZ], s[rT]
.endm

; ---- entry -------------------------------------------------------------------
  s_mov_b32 s[rA], %2
  s_mov_b32 s[rX], %3
  s_mov_b32 s[rY], %4
  s_mov_b32 s[rSP], %5
  s_mov_b32 s[rP], %6
  s_mov_b32 s[rIO], %7
  s_mov_b32 s[rFL], %8
  s_mov_b32 s[rVec], %13
  s_mov_b32 s[rL], %1
  s_mov_b64 exec, 1
  v_mov_b32 v[vL], %1
  v_mov_b32 v[vRAM], %12
  v_mov_b32 v[vRG], %14
  v_mov_b32 v[vZ], 0
  v_mov_b32 v[vF], %0
  v_mov_b32 v[v7FF], 0x7ff
  s_mov_b32 s[rLim], LIM
  s_movk_i32 s[rFF], 0xff
  s_movk_i32 s[r2000], 0x2000
  s_mov_b32 s[r2G], 0x20000000
  s_mov_b32 s[rLo], 0x80010
  s_mov_b32 s[rSel0], 0x0201000C
  s_mov_b32 s[rSel1], 0x0302010C
  s_mov_b32 s[rSel2], 0x0403020C
  s_mov_b32 s[rSel3], 0x0504030C
  s_getpc_b64 s[rRet:rRet+1]
.Lw%=_here:
  s_add_u32 s[rRet], s[rRet], .Lw%=_end-.Lw%=_here
  s_addc_u32 s[rRet+1], s[rRet+1], 0
  s_getpc_b64 s[rJ:rJ+1]
  s_add_u32 s[rJ], s[rJ], .Lw%=_table@rel32@lo+4
  s_addc_u32 s[rJ+1], s[rJ+1], .Lw%=_table@rel32@hi+12
  s_mov_b32 s[rTab], s[rJ]
  s_mov_b32 s[rQ], s[rJ]
  s_sub_u32 s[rExit], s[rJ], 0x10000
  UNPACK
  s_and_b32 s[rT], s[rTab], 0xFFFF
.if SOLO
  s_cbranch_scc1 .Lw%=_unfit
  s_cmp_eq_u32 s[rTab], 0   ; the exit table would lie in the 4 GB below
.endif
  s_cbranch_scc0 .Lw%=_start
.Lw%=_unfit:
  PACK                      ; a table that jumps do not reach: nothing runs here
  s_mov_b32 s[rK], 0
  s_mov_b32 s[rU], %0
  s_mov_b64 exec, -1
  s_branch .Lw%=_end
.Lw%=_start:
  ENTER vF
  ENTERED
.Lw%=_end:
  s_mov_b32 %0, s[rU]
  s_mov_b32 %1, s[rL]
  s_mov_b32 %2, s[rA]
  s_mov_b32 %3, s[rX]
  s_mov_b32 %4, s[rY]
  s_mov_b32 %5, s[rSP]
  s_mov_b32 %6, s[rT]
  s_mov_b32 %7, s[rIO]
  s_mov_b32 %8, s[rFL]
  s_mov_b32 %9, s[rK]
  s_mov_b32 %10, s[rR]
  s_mov_b32 %11, s[rM]

.pushsection .text.nes_wave, "ax", @progbits
.p2align 16
.if SOLO
.rept 256
.p2align 8
  s_branch .Lw%=_done
.endr
.p2align 16
.endif
.Lw%=_table:
; $00 BRK: return address and P|B|U at SP-2..SP, I set, to the vector
  H
  s_cmp_lt_u32 s[rSP], 2
  s_cbranch_scc1 .Lw%=_general
  s_cmp_eq_u32 s[rVec], 0
  s_cbranch_scc1 .Lw%=_general
  PACK
  s_or_b32 s[rT], s[rT], 16
  HERE rU, 2
  v_or_b32 v[vA], s[rSP], v[vRAM]
  v_mov_b32 v[vD], s[rU]
  ds_write_b16 v[vA], v[vD] offset:255
  v_mov_b32 v[vD], s[rT]
  ds_write_b8 v[vA], v[vD] offset:254
  s_sub_u32 s[rSP], s[rSP], 3
  s_and_b32 s[rSP], s[rSP], s[rFF]
  s_bitset1_b32 s[rP], 2
  s_mov_b32 s[rU], s[rVec]
  v_mov_b32 v[vA], s[rU]
  ENTER vA
  JUMP 21
  R_INDX ORA, rA
  ILL
.Lw%=_done:
  s_branch .Lw%=_exit
  ILL 2
  R_ZP ORA, rA
  M_ZP ASL
  ILL
; $08 PHP
  H
  AHEAD 1
  PACK
  s_or_b32 s[rT], s[rT], 16
  v_or_b32 v[vA], s[rSP], v[vRAM]
  v_mov_b32 v[vD], s[rT]
  ds_write_b8 v[vA], v[vD] offset:256
  s_sub_u32 s[rSP], s[rSP], 1
  s_and_b32 s[rSP], s[rSP], s[rFF]
  NEXT 9
  R_IMM ORA, rA
  A_ ASL, rA
  ILL 2
  R_ABS ORA, rA
  M_ABS ASL
  ILL
; $10
  BRANCH 0, s_and_b32 s[rT], s[rNZ], 0x8080
  R_INDY ORA, rA
  ILL 3
  R_ZPI ORA, rA, rX
  M_ZPX ASL
  ILL
  F_ s_mov_b32 s[rC], 0
  R_ABSI ORA, rA, rY
  ILL 3
  R_ABSI ORA, rA, rX
  M_ABSX ASL
  ILL
; $20 JSR: return address - 1 at SP-1, SP
  H
  s_cmp_eq_u32 s[rSP], 0
  s_cbranch_scc1 .Lw%=_general
  s_lshr_b32 s[rT], s[rW], 16
  TARGET vT, 16
  HERE rT, 2
  v_or_b32 v[vA], s[rSP], v[vRAM]
  v_mov_b32 v[vD], s[rT]
  ds_write_b16 v[vA], v[vD] offset:255
  s_sub_u32 s[rSP], s[rSP], 2
  s_and_b32 s[rSP], s[rSP], s[rFF]
  JUMP 18
  R_INDX AND, rA
  ILL 2
  R_ZP BIT, rA
  R_ZP AND, rA
  M_ZP ROL
  ILL
; $28 PLP
  H
  s_add_u32 s[rSP], s[rSP], 1
  s_and_b32 s[rSP], s[rSP], s[rFF]
  v_or_b32 v[vA], s[rSP], v[vRAM]
  ds_read_u8 v[vM], v[vA] offset:256
  AHEAD 1, 1
  s_waitcnt lgkmcnt(1)
  v_readfirstlane_b32 s[rP], v[vM]
  s_and_b32 s[rP], s[rP], 0xCF
  UNPACK
  NEXT 12
  R_IMM AND, rA
  A_ ROL, rA
  ILL
  R_ABS BIT, rA
  R_ABS AND, rA
  M_ABS ROL
  ILL
; $30
  BRANCH 1, s_and_b32 s[rT], s[rNZ], 0x8080
  R_INDY AND, rA
  ILL 3
  R_ZPI AND, rA, rX
  M_ZPX ROL
  ILL
  F_ s_mov_b32 s[rC], 1
  R_ABSI AND, rA, rY
  ILL 3
  R_ABSI AND, rA, rX
  M_ABSX ROL
  ILL
; $40 RTI: P, then the return address, from SP+1..SP+3
  H
  s_cmp_gt_u32 s[rSP], 0xFC
  s_cbranch_scc1 .Lw%=_general
  v_or_b32 v[vA], s[rSP], v[vRAM]
  ds_read_b32 v[vM], v[vA] offset:257
  s_waitcnt lgkmcnt(0)
  v_readfirstlane_b32 s[rM], v[vM]
  s_bfe_u32 s[rT], s[rM], 0x100008
  TARGET vM, 8
  v_mov_b32 v[vF], s[rU]
  s_add_u32 s[rSP], s[rSP], 3
  s_and_b32 s[rP], s[rM], 0xCF
  UNPACK
  PASS 18, .Lw%=_exit
  ENTERED
  R_INDX EOR, rA
  ILL 3
  R_ZP EOR, rA
  M_ZP LSR
  ILL
; $48 PHA
  H
  v_or_b32 v[vA], s[rSP], v[vRAM]
  v_mov_b32 v[vD], s[rA]
  ds_write_b8 v[vA], v[vD] offset:256
  AHEAD 1, 1
  s_sub_u32 s[rSP], s[rSP], 1
  s_and_b32 s[rSP], s[rSP], s[rFF]
  NEXT 9
  R_IMM EOR, rA
  A_ LSR, rA
  ILL
; $4C JMP: to itself is the idle loop, left to the general path
  H
  s_lshr_b32 s[rT], s[rW], 16
  TARGET vT, 16
  v_readfirstlane_b32 s[rM], v[vF]
  s_cmp_eq_u32 s[rU], s[rM]
  s_cbranch_scc1 .Lw%=_general
  JUMP 9
  R_ABS EOR, rA
  M_ABS LSR
  ILL
; $50
  BRANCHV 0
  R_INDY EOR, rA
  ILL 3
  R_ZPI EOR, rA, rX
  M_ZPX LSR
  ILL
  F_ s_bitset0_b32 s[rP], 2
  R_ABSI EOR, rA, rY
  ILL 3
  R_ABSI EOR, rA, rX
  M_ABSX LSR
  ILL
; $60 RTS
  H
  s_cmp_gt_u32 s[rSP], 0xFD
  s_cbranch_scc1 .Lw%=_general
  v_or_b32 v[vA], s[rSP], v[vRAM]
  ds_read_u16 v[vM], v[vA] offset:257
  s_waitcnt lgkmcnt(0)
  v_add_u32 v[vM], 1, v[vM]
  s_nop 0
  v_readfirstlane_b32 s[rT], v[vM]
  TARGET vM
  s_add_u32 s[rSP], s[rSP], 2
  JUMP 18
  R_INDX ADC, rA
  ILL 3
  R_ZP ADC, rA
  M_ZP ROR
  ILL
; $68 PLA
  H
  s_add_u32 s[rSP], s[rSP], 1
  s_and_b32 s[rSP], s[rSP], s[rFF]
  v_or_b32 v[vA], s[rSP], v[vRAM]
  ds_read_u8 v[vM], v[vA] offset:256
  AHEAD 1, 1
  s_waitcnt lgkmcnt(1)
  OP_LD rA
  NEXT 12
  R_IMM ADC, rA
  A_ ROR, rA
  ILL 2
  R_ABS ADC, rA
  M_ABS ROR
  ILL
; $70
  BRANCHV 1
  R_INDY ADC, rA
  ILL 3
  R_ZPI ADC, rA, rX
  M_ZPX ROR
  ILL
  F_ s_bitset1_b32 s[rP], 2
  R_ABSI ADC, rA, rY
  ILL 3
  R_ABSI ADC, rA, rX
  M_ABSX ROR
  ILL
; $80
  ILL
  W_INDX rA
  ILL 2
  W_ZP rY
  W_ZP rA
  W_ZP rX
  ILL
  A_ DEC, rY
  ILL
  T_ rA, rX
  ILL
  W_ABS rY
  W_ABS rA
  W_ABS rX
  ILL
; $90
  BRANCH 0, s_cmp_lg_u32 s[rC], 0
  W_INDY rA
  ILL 2
  W_ZPI rY, rX
  W_ZPI rA, rX
  W_ZPI rX, rY
  ILL
  T_ rA, rY
  W_ABSI rA, rY
  F_ s_mov_b32 s[rSP], s[rX]
  ILL 2
  W_ABSI rA, rX
  ILL 2
; $A0
  LD_IMM rY
  R_INDX LD, rA
  LD_IMM rX
  ILL
  R_ZP LD, rY
  R_ZP LD, rA
  R_ZP LD, rX
  ILL
  T_ rY, rA
  LD_IMM rA
  T_ rX, rA
  ILL
  R_ABS LD, rY
  R_ABS LD, rA
  R_ABS LD, rX
  ILL
; $B0
  BRANCH 1, s_cmp_lg_u32 s[rC], 0
  R_INDY LD, rA
  ILL 2
  R_ZPI LD, rY, rX
  R_ZPI LD, rA, rX
  R_ZPI LD, rX, rY
  ILL
  F_ s_mov_b32 s[rV1], 0
  R_ABSI LD, rA, rY
  T_ rX, rSP
  ILL
  R_ABSI LD, rY, rX
  R_ABSI LD, rA, rX
  R_ABSI LD, rX, rY
  ILL
; $C0
  R_IMM CP, rY
  R_INDX CP, rA
  ILL 2
  R_ZP CP, rY
  R_ZP CP, rA
  M_ZP DEC
  ILL
  A_ INC, rY
  R_IMM CP, rA
  A_ DEC, rX
  ILL
  R_ABS CP, rY
  R_ABS CP, rA
  M_ABS DEC
  ILL
; $D0
  BRANCH 1, s_and_b32 s[rT], s[rNZ], s[rFF]
  R_INDY CP, rA
  ILL 3
  R_ZPI CP, rA, rX
  M_ZPX DEC
  ILL
  F_ s_bitset0_b32 s[rP], 3
  R_ABSI CP, rA, rY
  ILL 3
  R_ABSI CP, rA, rX
  M_ABSX DEC
  ILL
; $E0
  R_IMM CP, rX
  R_INDX SBC, rA
  ILL 2
  R_ZP CP, rX
  R_ZP SBC, rA
  M_ZP INC
  ILL
  A_ INC, rX
  R_IMM SBC, rA
  F_ s_nop 0
  ILL
  R_ABS CP, rX
  R_ABS SBC, rA
  M_ABS INC
  ILL
; $F0
  BRANCH 0, s_and_b32 s[rT], s[rNZ], s[rFF]
  R_INDY SBC, rA
  ILL 3
  R_ZPI SBC, rA, rX
  M_ZPX INC
  ILL
  F_ s_bitset1_b32 s[rP], 3
  R_ABSI SBC, rA, rY
  ILL 3
  R_ABSI SBC, rA, rX
  M_ABSX INC
  ILL
.org .Lw%=_table+65536
.subsection 1

; ---- I/O registers programs poll: rT the address, the byte to rM -----------------
.Lw%=_ioread:
  s_cmp_eq_u32 s[rT], 0x2002
  s_cbranch_scc1 .Lw%=_ppustatus
  s_cmp_eq_u32 s[rT], 0x2004
  s_cbranch_scc1 .Lw%=_oamdata
  s_cmp_eq_u32 s[rT], 0x4016
  s_cbranch_scc1 .Lw%=_pad1
  s_branch .Lw%=_general
; PPUSTATUS: flags over the open bus's low bits; clears vblank, the pending
; NMI and the write toggle (io bits 0-7 open bus, 8-15 status).
.Lw%=_ppustatus:
  s_bfe_u32 s[rU], s[rW], 0x80008
  s_cmp_eq_u32 s[rU], 0xAD
  s_cbranch_scc1 .Lw%=_poll
  s_cmp_eq_u32 s[rU], 0x2C
  s_cbranch_scc1 .Lw%=_poll
.Lw%=_status:
  s_lshr_b32 s[rM], s[rIO], 8
  s_and_b32 s[rM], s[rM], 0xE0
  s_and_b32 s[rT], s[rIO], 0x1F
  s_or_b32 s[rM], s[rM], s[rT]
  s_andn2_b32 s[rIO], s[rIO], 0x80FF
  s_or_b32 s[rIO], s[rIO], s[rM]
  s_andn2_b32 s[rFL], s[rFL], 0x12
  s_setpc_b64 s[rCall:rCall+1]
; LDA or BIT $2002 of a loop that waits for a flag (a branch back to it next,
; or an AND between them): the general path skips to the next event.
.Lw%=_poll:
  s_waitcnt lgkmcnt(0)
  v_readfirstlane_b32 s[rR], v[vW]
  v_readfirstlane_b32 s[rU], v[vW+1]
  s_lshr_b32 s[rR], s[rR], 24
  s_cmp_eq_u32 s[rR], 0x29
  s_cbranch_scc1 .Lw%=_poll3
  s_and_b32 s[rR], s[rR], 0x1F
  s_cmp_lg_u32 s[rR], 0x10
  s_cbranch_scc1 .Lw%=_status
  s_and_b32 s[rR], s[rU], s[rFF]
  s_cmp_eq_u32 s[rR], 0xFB
  s_cbranch_scc1 .Lw%=_general
  s_branch .Lw%=_status
.Lw%=_poll3:
  s_bitcmp0_b32 s[rW], 15             ; LDA
  s_cbranch_scc1 .Lw%=_status
  s_bfe_u32 s[rR], s[rU], 0x50008
  s_cmp_lg_u32 s[rR], 0x10
  s_cbranch_scc1 .Lw%=_status
  s_bfe_u32 s[rR], s[rU], 0x80010
  s_cmp_eq_u32 s[rR], 0xF9
  s_cbranch_scc1 .Lw%=_general
  s_branch .Lw%=_status
; OAMDATA: the byte at OAMADDR, kept in flags bits 16-23.
.Lw%=_oamdata:
  s_bfe_u32 s[rM], s[rFL], 0x80010
  s_setpc_b64 s[rCall:rCall+1]
; Pad 1 (strobe low): the next button, then ones (io bits 16-23 shift
; register, 24-27 reads).
.Lw%=_pad1:
  s_bitcmp1_b32 s[rFL], 5
  s_cbranch_scc1 .Lw%=_general
  s_bitcmp1_b32 s[rIO], 27
  s_cbranch_scc1 .Lw%=_padout
  s_bfe_u32 s[rM], s[rIO], 0x10010
  s_or_b32 s[rM], s[rM], 64
  s_bfe_u32 s[rT], s[rIO], 0x70011
  s_lshl_b32 s[rT], s[rT], 16
  s_andn2_b32 s[rIO], s[rIO], 0xFF0000
  s_or_b32 s[rIO], s[rIO], s[rT]
  s_add_u32 s[rIO], s[rIO], 0x1000000
  s_setpc_b64 s[rCall:rCall+1]
.Lw%=_padout:
  s_movk_i32 s[rM], 0x41
  s_setpc_b64 s[rCall:rCall+1]

; ---- stores to I/O registers: rT the address, rM the byte -------------------------
; The ones programs make in numbers; the instruction is otherwise done, the
; next one's window on its way.  The rest leave the block.  (vcc holds the
; countdown's borrow throughout where SOLO is 0.)
.Lw%=_store:
  s_cmp_eq_u32 s[rT], 0x2007
  s_cbranch_scc1 .Lw%=_ppudata
  s_sub_u32 s[rU], s[rT], 0x4000
  s_cmp_le_u32 s[rU], 0x16
  s_cbranch_scc1 .Lw%=_apu
  s_cmp_eq_u32 s[rT], 0x2006
  s_cbranch_scc1 .Lw%=_ppuaddr
  s_cmp_eq_u32 s[rT], 0x2005
  s_cbranch_scc1 .Lw%=_ppuscroll
  s_cmp_eq_u32 s[rT], 0x2001
  s_cbranch_scc1 .Lw%=_ppumask
  s_cmp_eq_u32 s[rT], 0x2000
  s_cbranch_scc1 .Lw%=_ppuctrl
.Lw%=_other:
  s_mov_b32 s[rR], s[rT]
  s_mov_b32 s[rK], 2
  s_branch .Lw%=_leave
.macro RESUME
.if SOLO == 0
  s_cbranch_vccnz .Lw%=_exit
.endif
  AIM
  GO
.endm
.macro OPENBUS
  s_andn2_b32 s[rIO], s[rIO], 0xFF
  s_or_b32 s[rIO], s[rIO], s[rM]
.endm
; $4000-$4016 but $4014: the byte kept for reads; $4016 is the pads' strobe
; too (high or on its way down it loads pad 1's buttons and clears the counts
; of reads: flags bits 5 and 8-15, io bits 16-31).
.Lw%=_apu:
  s_cmp_eq_u32 s[rU], 0x14
  s_cbranch_scc1 .Lw%=_other
  ds_read_b64 v[vP:vP+1], v[vRG] offset:48
  ds_read_b32 v[vD], v[vRG] offset:56
  s_waitcnt lgkmcnt(0)
  v_readfirstlane_b32 s[rCall], v[vP]
  v_readfirstlane_b32 s[rCall+1], v[vP+1]
  v_readfirstlane_b32 s[rR], v[vD]
  s_cmp_lg_u32 s[rU], 0x16
  s_mul_i32 s[rU], s[rU], s[rR]
  s_cbranch_scc1 .Lw%=_apubyte
  s_bfe_u32 s[rT], s[rFL], 0x80008
  s_lshl_b32 s[rT], s[rT], 16
  s_and_b32 s[rR], s[rIO], 0xFFFF
  s_or_b32 s[rT], s[rT], s[rR]
  s_bfe_u32 s[rR], s[rFL], 0x10005
  s_or_b32 s[rR], s[rR], s[rM]
  s_bitcmp1_b32 s[rR], 0
  s_cselect_b32 s[rIO], s[rT], s[rIO]
  s_andn2_b32 s[rFL], s[rFL], 32
  s_and_b32 s[rT], s[rM], 1
  s_lshl_b32 s[rT], s[rT], 5
  s_or_b32 s[rFL], s[rFL], s[rT]
.Lw%=_apubyte:
  v_mov_b32 v[vD], s[rM]
  s_add_u32 s[rCall], s[rCall], s[rU]
  s_addc_u32 s[rCall+1], s[rCall+1], 0
  global_store_byte v[vZ], v[vD], s[rCall:rCall+1]
  RESUME
; PPUDATA to the nametables (palette and CHR leave): the byte at v, v past it.
.Lw%=_ppudata:
  ds_read_u16 v[vM], v[vRG] offset:16
  ds_read_b32 v[vD], v[vRG] offset:60
  ds_read_b64 v[vP:vP+1], v[vRG] offset:40
  s_waitcnt lgkmcnt(0)
  v_readfirstlane_b32 s[rU], v[vM]
  v_readfirstlane_b32 s[rR], v[vD]
  v_readfirstlane_b32 s[rCall], v[vP]
  v_readfirstlane_b32 s[rCall+1], v[vP+1]
  s_and_b32 s[rJ], s[rU], 0x3FFF
  s_sub_u32 s[rJ], s[rJ], 0x2000
  s_cmp_ge_u32 s[rJ], 0x1F00
  s_cbranch_scc1 .Lw%=_other
  s_and_b32 s[rK], s[rJ], s[rR]        ; mirroring: two masks (kWaveNt)
  s_lshr_b32 s[rJ], s[rJ], 1
  s_lshr_b32 s[rR], s[rR], 16
  s_and_b32 s[rJ], s[rJ], s[rR]
  s_or_b32 s[rK], s[rK], s[rJ]
  s_add_u32 s[rCall], s[rCall], s[rK]
  s_addc_u32 s[rCall+1], s[rCall+1], 0
  ds_read_u8 v[vM], v[vRG]
  v_mov_b32 v[vD], s[rM]
  global_store_byte v[vZ], v[vD], s[rCall:rCall+1]
  OPENBUS
  s_waitcnt lgkmcnt(0)
  v_readfirstlane_b32 s[rR], v[vM]
  s_bitcmp1_b32 s[rR], 2
  s_cselect_b32 s[rR], 32, 1
  s_add_u32 s[rU], s[rU], s[rR]
  v_mov_b32 v[vD], s[rU]
  ds_write_b16 v[vRG], v[vD] offset:16
  RESUME
; PPUADDR: t's high byte, then its low byte and v.
.Lw%=_ppuaddr:
  ds_read_u16 v[vM], v[vRG] offset:18
  OPENBUS
  s_xor_b32 s[rFL], s[rFL], 16
  s_waitcnt lgkmcnt(0)
  v_readfirstlane_b32 s[rU], v[vM]
  s_bitcmp1_b32 s[rFL], 4
  s_cbranch_scc0 .Lw%=_ppuaddr2
  s_and_b32 s[rU], s[rU], s[rFF]
  s_and_b32 s[rR], s[rM], 0x3F
  s_lshl_b32 s[rR], s[rR], 8
  s_or_b32 s[rU], s[rU], s[rR]
  v_mov_b32 v[vD], s[rU]
  ds_write_b16 v[vRG], v[vD] offset:18
  RESUME
.Lw%=_ppuaddr2:
  s_and_b32 s[rU], s[rU], 0x7F00
  s_or_b32 s[rU], s[rU], s[rM]
  v_mov_b32 v[vD], s[rU]
  ds_write_b16 v[vRG], v[vD] offset:18
  ds_write_b16 v[vRG], v[vD] offset:16
  RESUME
; PPUMASK.
.Lw%=_ppumask:
  OPENBUS
  v_mov_b32 v[vD], s[rM]
  ds_write_b8 v[vRG], v[vD] offset:1
  RESUME
; PPUCTRL: t's nametable too; turning NMI on during vblank raises one, which
; the kernel takes.
.Lw%=_ppuctrl:
  ds_read_u8 v[vA], v[vRG]
  ds_read_u16 v[vM], v[vRG] offset:18
  s_waitcnt lgkmcnt(0)
  v_readfirstlane_b32 s[rR], v[vA]
  v_readfirstlane_b32 s[rU], v[vM]
  s_andn2_b32 s[rR], s[rM], s[rR]
  s_lshr_b32 s[rK], s[rIO], 8
  s_and_b32 s[rR], s[rR], s[rK]
  s_bitcmp1_b32 s[rR], 7
  s_cbranch_scc1 .Lw%=_other
  OPENBUS
  s_and_b32 s[rU], s[rU], 0xF3FF
  s_and_b32 s[rR], s[rM], 3
  s_lshl_b32 s[rR], s[rR], 10
  s_or_b32 s[rU], s[rU], s[rR]
  v_mov_b32 v[vA], s[rM]
  v_mov_b32 v[vD], s[rU]
  ds_write_b8 v[vRG], v[vA]
  ds_write_b16 v[vRG], v[vD] offset:18
  RESUME
; PPUSCROLL: x (fine x, t's coarse x), then y (t's coarse and fine y).
.Lw%=_ppuscroll:
  ds_read_u16 v[vM], v[vRG] offset:18
  OPENBUS
  s_xor_b32 s[rFL], s[rFL], 16
  s_waitcnt lgkmcnt(0)
  v_readfirstlane_b32 s[rU], v[vM]
  v_mov_b32 v[vA], s[rM]
  s_bitcmp1_b32 s[rFL], 4
  s_cbranch_scc0 .Lw%=_ppuscroll2
  ds_write_b8 v[vRG], v[vA] offset:8
  v_and_b32 v[vA], 7, v[vA]
  ds_write_b8 v[vRG], v[vA] offset:6
  s_and_b32 s[rU], s[rU], 0xFFE0
  s_lshr_b32 s[rR], s[rM], 3
  s_or_b32 s[rU], s[rU], s[rR]
  v_mov_b32 v[vD], s[rU]
  ds_write_b16 v[vRG], v[vD] offset:18
  RESUME
.Lw%=_ppuscroll2:
  ds_write_b8 v[vRG], v[vA] offset:9
  s_and_b32 s[rU], s[rU], 0x8C1F
  s_and_b32 s[rR], s[rM], 7
  s_lshl_b32 s[rR], s[rR], 12
  s_or_b32 s[rU], s[rU], s[rR]
  s_and_b32 s[rR], s[rM], 0xF8
  s_lshl_b32 s[rR], s[rR], 2
  s_or_b32 s[rU], s[rU], s[rR]
  v_mov_b32 v[vD], s[rU]
  ds_write_b16 v[vRG], v[vD] offset:18
  RESUME

; ---- exits -------------------------------------------------------------------
.Lw%=_exit:
  s_mov_b32 s[rK], 1
  s_branch .Lw%=_leave
; A taken branch that leaves the image: the PC back at it, from vD past it.
.Lw%=_back:
  v_subrev_u32 v[vF], 2, v[vD]
.Lw%=_general:
  s_mov_b32 s[rK], 0
.Lw%=_leave:
  s_waitcnt vmcnt(0) lgkmcnt(0)
.if SOLO == 0
  v_readfirstlane_b32 s[rL], v[vL]
.endif
  PACK
  v_readfirstlane_b32 s[rU], v[vF]
  s_mov_b64 exec, -1
  s_setpc_b64 s[rRet:rRet+1]
.subsection 0
.popsection
)"
        : "+s"(pc), "+s"(left), "+s"(a), "+s"(x), "+s"(y), "+s"(sp), "+s"(p), "+s"(io), "+s"(fl), "=&s"(why), "=&s"(addr),
          "=&s"(value)
        : "s"(ram), "s"(vec), "s"(regs)
        : "memory", "scc", "vcc", "s34", "s35", "s36", "s37", "s38", "s39", "s40", "s41", "s42", "s43", "s44",
          "s45", "s46", "s47", "s48", "s49", "s50", "s51", "s52", "s53", "s54", "s55", "s56", "s57", "s58", "s59",
          "s60", "s61", "s62", "s63", "s64", "s65", "s66", "s67", "s68", "s69", "s70",
          "v8", "v9", "v10", "v11", "v12", "v13",
          "v14", "v15", "v16", "v17", "v18", "v19", "v20", "v22", "v23");
    c.pc = (pc - kWaveRom + 0x8000u) & 0xFFFFu;
    c.left = static_cast<std::int32_t>(left + 1u);
    c.a = a; c.x = x; c.y = y; c.sp = sp; c.p = p;
    c.io = io; c.flags = fl;
    c.addr = addr; c.value = value;
    return why;
}

}  // namespace nesle
