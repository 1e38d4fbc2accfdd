// nes_step_wave.hip -- the step kernel with one console per wave, for batches
// too small to fill the lanes of the chip's waves.
//
// A wave of the step kernel (nes_step.hip) takes about 1,060 cycles per
// emulated instruction however few consoles it serves: at 4,096 consoles 60
// of 64 lanes idle, and a single console takes as long as 8,192.  Here a wave
// runs one console on the scalar unit, each opcode by its own code
// (nes_wave.h), about 165 cycles per instruction alone on a SIMD and 30 per
// SIMD with eight waves on it.  Frame-skip 4, the workload ROM, ms per launch
// (lane kernel -> this one): 1 console 13.0 -> 2.13, 1,000 13.4 -> 2.46,
// 4,096 13.8 -> 2.73, 8,192 14.1 -> 3.37, 16,384 16.7 -> 6.51, 32,768
// 17.3 -> 12.9.
//
// What the block of assembly leaves to the general path here -- I/O and PRG
// RAM, NMI entry, code outside PRG ROM, PPU events, OAM DMA, frame capture --
// uses the lane kernel's own routines (nes_step.hip), every lane doing the
// same for the wave's console.
//
// A workgroup is up to 16 waves around one copy of the PRG image.  Two of
// them share a CU (eight waves per SIMD): 67,584 bytes of LDS each, and at
// most 80 scalar registers per wave (a SIMD's 800 are handed out by 16; with
// 96 only seven waves fit and the second workgroup waits for the first:
// 8,192 consoles 6.9 ms instead of 5.1 when it was so).
//
// Statistics and binding instruction budgets stay with the lane kernel, as do
// images whose flow can run past their end, and programs that take the general
// path too often (nes_choice.h): an instruction there costs 1,100 to 1,700
// cycles of a SIMD, where a lane of the lane kernel shares 1,400 with 63
// others.
//
// Built twice: this file's own instance for many waves per SIMD, and
// nes_step_solo.hip's for few (SOLO in nes_wave.h).
#define NESLE_STEP_PART 3
#ifndef NESLE_WAVE_SOLO
#define NESLE_WAVE_SOLO "0"
#define NESLE_WAVE_KERNEL wave_kernel
#define NESLE_WAVE_LAUNCH launch_step_wave
#endif
#include "nes_step.hip"

#include "nes_wave.h"

namespace nesle {
namespace {

constexpr std::uint32_t kWaveMaxWaves = 16;
// LDS: guard, PRG image, guard (nes_wave.h), the consoles' register areas in
// the gap up to the first console's RAM, which is aligned to its size.
constexpr std::uint32_t kIllegalOpcode = 0x02;
constexpr std::uint32_t kWaveRegs = kWaveRom + kPrgRomMax + kWaveGuard;
constexpr std::uint32_t kWaveRam = 17 * kRamBytes;
static_assert(kWaveRom == kLdsRom && kWaveRegs + kWaveMaxWaves * kWaveRegsBytes <= kWaveRam, "LDS layout");
static_assert(kWaveRam + kWaveMaxWaves * kRamBytes == kLdsLimit, "LDS layout");

// A value every lane holds, in a scalar register.
__device__ __forceinline__ std::uint32_t uni(std::uint32_t v) { return __builtin_amdgcn_readfirstlane(v); }

// Priority by the time a console has left in the launch, in quarters.  A SIMD
// issues its oldest wave first, so of two workgroups on a CU the older runs
// ahead and the younger ends alone; with the ones behind first they end
// together.
__device__ __forceinline__ void yield(std::uint32_t frames_left, std::uint32_t dot, std::uint32_t frameskip) {
    const std::uint64_t all = static_cast<std::uint64_t>(frameskip) * kFrameDots;
    const std::uint64_t left4 = 4 * (static_cast<std::uint64_t>(frames_left) * kFrameDots - dot);
    if (left4 <= all) {
        __builtin_amdgcn_s_setprio(0);
    } else if (left4 <= 2 * all) {
        __builtin_amdgcn_s_setprio(1);
    } else if (left4 <= 3 * all) {
        __builtin_amdgcn_s_setprio(2);
    }
}

// A loop that waits for a PPUSTATUS flag: LDA or BIT $2002 at `pc`, which has
// just read `v`, an AND # or none, and a branch back.  The flags change only
// at PPU events and with the read itself (it clears bit 7, and the open bus
// then holds what it read), so once bit 7 is clear every pass leaves the
// registers as the one before, and the passes that end before the next event,
// `left` dots away, are skipped: their dots are returned.
__device__ __forceinline__ std::uint32_t waited(std::uint32_t pc, std::uint32_t v, std::uint32_t p, std::int32_t left) {
    if (v & 0x80) return 0;
    const std::uint8_t* at = lds + kLdsRom + (pc & 0x7FFF) + 3;
    const std::uint32_t b0 = uni(at[0]), b1 = uni(at[1]), b2 = uni(at[2]), b3 = uni(at[3]);
    const bool masked = b0 == 0x29;
    const std::uint32_t op = masked ? b2 : b0, rel = masked ? b3 : b1, len = masked ? 7u : 5u;
    if ((op & 0x1F) != 0x10 || rel != 0x100 - len) return 0;
    if (masked) {   // the flags the AND leaves, of A (BIT does not load it: such a loop is not skipped)
        if (uni(at[-3]) != 0xAD) return 0;
        const std::uint32_t r = v & b1;
        p = (p & ~0x82u) | (r & 0x80) | (r == 0 ? 2u : 0u);
    }
    const std::uint32_t* d = c_micro_full.e[op].d;
    if (ubfe(p ^ ((d[2] >> 8) & 0xFF), d[2], d[3]) == 0) return 0;   // falls through
    const std::uint32_t cross = (((pc + len) ^ pc) & 0xFF00) ? 1u : 0u;
    const std::uint32_t pass = 3 * (4 + (masked ? 2 : 0) + 3 + cross);
    return (static_cast<std::uint32_t>(left) - 1) / pass * pass;
}

__global__ void __launch_bounds__(64 * kWaveMaxWaves) __attribute__((amdgpu_num_sgpr(80)))
NESLE_WAVE_KERNEL(DeviceState s, std::uint32_t frameskip) {
    using C = Console<true>;
    const std::uint32_t tid = threadIdx.x, lane = tid & 63, T = blockDim.x, W = T >> 6;
    const std::uint32_t wave = uni(tid >> 6);
    const std::uint32_t env0 = xcd_block(blockIdx.x, gridDim.x) * W;
    const std::uint32_t env = env0 + wave;
    const std::uint32_t P = s.pitch;
    const bool mine = env < s.n;

    const bool lanes = s.choice->next != 0;   // the lane kernel behind takes this step
    if (blockIdx.x == 0 && tid == 0) s.choice->now = lanes ? 1u : 0u;
    if (lanes) return;

    {   // PRG ROM (a 16 KB image mirrored to 32 KB) between its guards.
        const std::uint32_t words = (s.prg_mask + 1) / 16;
        const uint4* src = reinterpret_cast<const uint4*>(s.prg_rom);
        uint4* dst = reinterpret_cast<uint4*>(lds + kLdsRom);
        for (std::uint32_t i = tid; i < kPrgRomMax / 16; i += T) dst[i] = src[i & (words - 1)];
        for (std::uint32_t i = tid; i < kWaveGuard; i += T) {
            lds[kLdsRom - kWaveGuard + i] = kIllegalOpcode;
            lds[kLdsRom + kPrgRomMax + i] = kIllegalOpcode;
        }
    }
    // RAM rows of the workgroup's consoles, adjacent bytes of a row, four
    // consoles at a time where there are four (env0 is then a multiple of
    // four, as the pitch is; the last workgroup's consoles may end past the
    // pitch).
    if (W >= 4) {
        for (std::uint32_t q = 0; q < W && env0 + q < P; q += 4) {
            for (std::uint32_t row = tid; row < kRamBytes; row += T) {
                const std::uint32_t v =
                    *reinterpret_cast<const std::uint32_t*>(s.ram + static_cast<std::size_t>(row) * P + env0 + q);
                std::uint8_t* at = lds + kWaveRam + q * kRamBytes + row;
                at[0] = static_cast<std::uint8_t>(v);
                at[kRamBytes] = static_cast<std::uint8_t>(v >> 8);
                at[2 * kRamBytes] = static_cast<std::uint8_t>(v >> 16);
                at[3 * kRamBytes] = static_cast<std::uint8_t>(v >> 24);
            }
        }
    } else {
        for (std::uint32_t q = 0; q < W; ++q)
            for (std::uint32_t row = tid; row < kRamBytes; row += T)
                lds[kWaveRam + q * kRamBytes + row] = s.ram[static_cast<std::size_t>(row) * P + env0 + q];
    }
    __syncthreads();

    const std::uint32_t base = kWaveRam + wave * kRamBytes;
    C c{(KState*)__builtin_amdgcn_kernarg_segment_ptr(), env, base, P};
    c.regs_base = kWaveRegs + wave * kWaveRegsBytes;
    const std::uint32_t brk = uni(lds[kLdsRom + 0x7FFE] | (lds[kLdsRom + 0x7FFF] << 8));
    WaveCpu cpu{};
    std::uint32_t fd0 = 0, flags = 0, frames = 0;
    if (mine) {
        c.w8(reg::kCtrl, s.ctrl[env]); c.w8(reg::kMask, s.mask[env]);
        c.w8(reg::kOamAddr, s.oam_addr[env]);
        c.w8(reg::kReadBuffer, s.read_buffer[env]); c.w8(reg::kFineX, s.fine_x[env]);
        c.w8(reg::kScrollX, s.scroll_x[env]); c.w8(reg::kScrollY, s.scroll_y[env]);
        c.w16(reg::kV, s.v[env]); c.w16(reg::kT, s.t[env]);
        {   // what the assembly's I/O stores need
            auto put64 = [&](std::uint32_t at, const std::uint8_t* v) {
                *reinterpret_cast<std::uint64_t*>(lds + c.regs_base + at) = reinterpret_cast<std::uint64_t>(v);
            };
            put64(kWaveVram, c.vmem() + vram::kNametable);
            put64(kWaveApu, s.apu_io + env);
            c.w32(kWavePitch, P);
            c.w32(kWaveNt, s.nt_mode == 2 ? 0xFFFu : s.nt_mode == 0 ? 0x7FFu : 0x3FFu | (0x400u << 16));
            static_assert(reg::kCtrl == 0 && reg::kFineX == 6 && reg::kScrollX == 8 && reg::kScrollY == 9 &&
                              reg::kV == 16 && reg::kT == 18 && reg::kBudgetHits + 4 <= kWaveVram,
                          "register area as nes_wave.h reads it");
        }
        fd0 = uni(s.frame_dot[env]);
        const std::uint32_t horizon0 = to_event(fd0, frameskip > 1);
        c.w32(reg::kFrameDot, fd0);
        c.w32(reg::kHorizon, horizon0);
        // The pad reads this step's mask; a high strobe re-latches (controller.hpp:20-25).
        const std::uint32_t buttons = s.actions[env], strobe = s.strobe[env];
        c.io = uni(s.open_bus[env] | (s.status[env] << 8) | ((strobe ? buttons : s.c1_shift[env]) << 16) |
                   ((strobe ? 0u : s.c1_count[env] & 0xFu) << 24) | (static_cast<std::uint32_t>(s.c2_count[env] & 0xF) << 28));
        c.flags = (s.nmi_pending[env] ? kNmiPending : 0u) | (s.fault[env] ? kFault : 0u) | (s.w[env] ? kWToggle : 0u) |
                  (strobe ? kStrobeBit : 0u) | (buttons << 8);
        c.set_oam_data(c.vmem()[vram::kOam + s.oam_addr[env]]);
        c.flags = uni(c.flags);
        c.w32(reg::kFramesLeft, (c.flags & kFault) ? 0u : frameskip);
        c.w32(reg::kFrames, 0);
        cpu.pc = uni(s.pc[env]);
        cpu.a = uni(s.a[env]); cpu.x = uni(s.x[env]); cpu.y = uni(s.y[env]);
        cpu.sp = uni(s.sp[env]); cpu.p = uni(s.p[env]);
        cpu.left = static_cast<std::int32_t>(uni(horizon0));
        __builtin_amdgcn_s_setprio(3);
        std::uint32_t general = 0, jumps = 0;   // trips through the general path, jumps of idle loops
        bool active = !(c.flags & kFault) && frameskip != 0;
        while (active) {
            const bool nmi = (c.flags & kNmiPending) != 0;
            bool counted = true;
            std::uint32_t dots = 0;
            std::uint32_t why = kWaveGeneral;
            if (!nmi && cpu.pc - 0x8000u < kWaveRomEnd && cpu.left > 0) {
                cpu.io = c.io;
                cpu.flags = c.flags;
                why = wave_run(cpu, base, c.regs_base, brk);
                c.io = cpu.io;
                c.flags = cpu.flags;
            }
            c.s = reload(c.s);
            general += why != kWaveEvent ? 1u : 0u;
            if (why == kWaveStore) {
                const std::uint32_t at = cpu.addr & 0xFFFF;
                if (at < 0x2000) {
                    lds[base + (at & 0x7FF)] = static_cast<std::uint8_t>(cpu.value);
                } else if (at < 0x8000) {
                    cpu.left -= static_cast<std::int32_t>(uni(c.io_wr(at, cpu.value)));
                }
            } else if (why == kWaveGeneral) {
                // One instruction (or the NMI entry) from the microcode, every
                // access through the bus.
                const std::uint32_t pc0 = cpu.pc, p0 = cpu.p, sp = cpu.sp;
                std::uint32_t mi = mc::kNmiEntry, b1 = 0, b2 = 0;
                if (!nmi) {
                    mi = uni(c.bus_rd(pc0));
                    const std::uint32_t len = (c_micro_full.e[mi].d[0] >> 12) & 3;
                    if (len >= 2) b1 = uni(c.bus_rd((pc0 + 1) & 0xFFFF));
                    if (len >= 3) b2 = uni(c.bus_rd((pc0 + 2) & 0xFFFF));
                }
                const std::uint32_t* d = c_micro_full.e[mi].d;
                const std::uint32_t d0 = d[0], d1 = d[1], d2 = d[2], d3 = d[3], d14 = d[14], d18 = d[18];
                const std::uint32_t regs0 = cpu.a | (cpu.x << 8) | (cpu.y << 16) | (sp << 24);
                const std::uint32_t abs = b1 | (b2 << 8);
                std::uint32_t ebase = abs;
                if (d0 & 0x20) {
                    const std::uint32_t pz = (b1 + (((mi & 0x1F) == 0x01) ? cpu.x : 0u)) & 0xFF;
                    ebase = uni(lds[base + pz] | (lds[base + ((pz + 1) & 0xFF)] << 8));
                }
                const std::uint32_t ea_full = ebase + ubfe(regs0, d0, d1);
                const std::uint32_t ea = ea_full & d[17];
                const std::uint32_t cross = ((ea_full ^ ebase) >> 8) & (d0 >> 7) & 1;
                const bool rd = d0 & 0x100, wr = d0 & 0x200;
                // Pulled bytes.
                const std::uint32_t v1 = lds[base + 0x100 + ((sp + 1) & 0xFF)], v2 = lds[base + 0x100 + ((sp + 2) & 0xFF)];
                const std::uint32_t v3 = lds[base + 0x100 + ((sp + 3) & 0xFF)];
                std::uint32_t M = b1;
                if (d[13] & 0xFF) M = uni(v1);
                if (rd) M = uni(c.bus_rd(ea));
                // Adder, logic unit and right shifter (nes_step.hip).
                const std::uint32_t R = ubfe(regs0, d2, 8);
                const std::uint32_t xa = sel(d18 & 0xFF, M, R);
                const std::uint32_t xb = (((d1 & 0x40) ? xa : M) & ((d1 >> 16) & 0xFF)) ^ (d1 >> 24);
                const std::uint32_t cf = p0 & 1;
                const std::uint32_t sum = xa + xb + ((cf & (d18 >> 8)) | ((d18 >> 16) & 1));
                const std::uint32_t lres = (R & M & ((d2 >> 8) & 0xFF)) | ((R ^ M) & ((d2 >> 16) & 0xFF));
                const std::uint32_t sr = (xa >> 1) | ((cf & (d1 >> 10)) << 7);
                const bool right = (d[19] & 0xFF) != 0;
                const std::uint32_t r = right ? sr : ((sum & (d2 >> 24)) | lres);
                const std::uint32_t carry = (right ? xa : sum >> 8) & 1;
                const std::uint32_t ovf = ((~(xa ^ xb) & (xa ^ sum)) >> 1) & 0x40;
                const std::uint32_t nv = (d0 & 0x800000) ? (M & 0xC0) : ((r & 0x80) | ovf);
                const std::uint32_t f = nv | (r == 0 ? 2u : 0u) | carry, fm = d0 >> 24;
                const std::uint32_t p1 = (((p0 & ~fm) | (f & fm)) & ((d3 >> 16) & 0xFF)) | (d3 >> 24);
                cpu.p = (d[15] & 0xFF) ? ((M & 0xCF) | 0x20) : p1;
                const std::uint32_t regs = sel(d[8], r << ((d3 >> 5) & 31), regs0) + d[6];
                // Next PC.
                const std::uint32_t fall = (pc0 + ((d0 >> 12) & 3)) & 0xFFFF;
                const std::uint32_t taken = ubfe(p0 ^ ((d2 >> 8) & 0xFF), d2, d3);
                const std::uint32_t target =
                    (fall + static_cast<std::uint32_t>(static_cast<std::int32_t>(static_cast<std::int8_t>(b1)))) & 0xFFFF;
                std::uint32_t next = taken ? target : fall;
                if (d[9]) next = abs;
                if (d[10]) next = uni((((v1 | (v2 << 8) | (v3 << 16)) >> (d[12] & 31)) + ((d[12] >> 16) & 1)) & 0xFFFF);
                if (d[11]) {
                    const std::uint32_t at = nmi ? 0x7FFA : 0x7FFE;
                    next = uni(lds[kLdsRom + at] | (lds[kLdsRom + at + 1] << 8));
                }
                if (d14 & mc::kJmpInd) {
                    next = uni(c.bus_rd(abs));
                    next |= uni(c.bus_rd((abs & 0xFF00) | ((abs + 1) & 0xFF))) << 8;
                }
                dots = 3 * ((d[16] >> 16) + cross + (taken ? (((fall ^ target) & 0xFF00) ? 2u : 1u) : 0u));
                // Pushes, then the operand write.
                if (d[4]) {
                    const std::uint32_t ret = pc0 + ((d[12] >> 24) & 3);
                    const std::uint32_t pb = (p0 & 0xEF) | ((d[15] >> 8) & 0xFF);
                    const std::uint32_t pw = __builtin_amdgcn_perm((regs0 << 8) | pb, ret, d[5]);
                    const std::uint32_t npush = (d[4] >> 16 & 1) + (d[4] >> 8 & 1) + (d[4] & 1);
                    for (std::uint32_t k = 0; k < npush; ++k)
                        lds[base + 0x100 + ((sp - k) & 0xFF)] = static_cast<std::uint8_t>(pw >> (8 * (2 - k)));
                }
                if (wr) {
                    if (ea < 0x2000) {
                        lds[base + (ea & 0x7FF)] = static_cast<std::uint8_t>(r);
                    } else if (ea < 0x8000) {
                        dots += c.io_wr(ea, r);
                    }
                }
                c.flags &= ~(d14 & mc::kClearNmi);
                counted = (d14 & mc::kCount) != 0;
                cpu.pc = next;
                cpu.a = regs & 0xFF; cpu.x = (regs >> 8) & 0xFF; cpu.y = (regs >> 16) & 0xFF; cpu.sp = regs >> 24;
                // Idle loop (JMP to itself): the jumps until the next event in one go.
                const std::int32_t gap = cpu.left - static_cast<std::int32_t>(dots);
                if ((d14 & mc::kJmpAbs) && abs == pc0 && gap > 0) {
                    const std::uint32_t skipped = uni(static_cast<std::uint32_t>((gap + 8) / 9));
                    dots += 9u * skipped;
                    jumps += skipped;
                }
                if (d14 & mc::kIllegal) {
                    c.flags |= kFault;
                    active = false;
                }
                cpu.left = static_cast<std::int32_t>(uni(static_cast<std::uint32_t>(cpu.left) - dots));
                if ((mi == 0xAD || mi == 0x2C) && ea == 0x2002 && cpu.left > 0 && pc0 - 0x8000u < kWaveRomEnd - 8u)
                    cpu.left -= static_cast<std::int32_t>(waited(pc0, M, cpu.p, cpu.left));
            }
            if (counted && cpu.left <= 0) {   // a timing event was crossed: settle the PPU
                const std::uint32_t fc = c.settle(c.r32(reg::kHorizon) - static_cast<std::uint32_t>(cpu.left), false);
                std::uint32_t fl = uni(c.r32(reg::kFramesLeft));
                if (uni(fc)) {
                    c.w32(reg::kFrames, c.r32(reg::kFrames) + 1);
                    fl -= 1;
                    c.w32(reg::kFramesLeft, fl);
                    if (fl == 0) active = false;
                }
                const std::uint32_t h = to_event(c.r32(reg::kFrameDot), fl > 1);
                c.w32(reg::kHorizon, h);
                cpu.left = static_cast<std::int32_t>(uni(h));
                yield(fl, uni(c.r32(reg::kFrameDot)), frameskip);
            }
            c.flags = uni(c.flags);
            c.io = uni(c.io);
            // OAM DMA (console.hpp:191-197): 256 bytes, 4 per lane; I/O pages
            // through the bus in order.
            if (c.flags & kDmaPending) {
                const std::uint32_t page = uni(c.r8(reg::kDmaPage)), oa = uni(c.r8(reg::kOamAddr));
                std::uint8_t* oam = c.s->vram + static_cast<std::size_t>(env) * c.s->vram_stride + vram::kOam;
                if (page < 0x20 || page >= 0x60) {
                    std::uint32_t val[4];
#pragma unroll
                    for (std::uint32_t k = 0; k < 4; ++k) {
                        const std::uint32_t addr = (page << 8) | (4 * lane + k);
                        if (page < 0x20) {
                            val[k] = lds[base + (addr & 0x7FF)];
                        } else if (page < 0x80) {
                            val[k] = c.s->ram[__umul24(addr - 0x5800, P) + env];
                        } else {
                            val[k] = lds[kLdsRom + (addr & 0x7FFF)];
                        }
                    }
#pragma unroll
                    for (std::uint32_t k = 0; k < 4; ++k) oam[(oa + 4 * lane + k) & 0xFF] = static_cast<std::uint8_t>(val[k]);
                    c.set_oam_data(uni(val[0]));   // OAM[OAMADDR] is now the page's first byte
                } else {
                    // OAMADDR advances with every byte (ppu.hpp:131-134), which a
                    // $2004 read inside the copy observes; it wraps back to `oa`.
                    std::uint32_t first = 0;
                    for (std::uint32_t i = 0; i < 256; ++i) {
                        const std::uint32_t at = (oa + i) & 0xFF;
                        c.w8(reg::kOamAddr, at);
                        c.set_oam_data(oam[at]);
                        const std::uint32_t val = c.bus_rd((page << 8) | i);
                        oam[at] = static_cast<std::uint8_t>(val);
                        if (i == 0) first = val;
                    }
                    c.w8(reg::kOamAddr, oa);
                    c.set_oam_data(first);
                }
                c.flags = uni(c.flags & ~kDmaPending);
                c.io = uni(c.io);
            }
            if (c.flags & kPresentPending) {
                C::capture(c.s, env, c.regs_base, lane, 64);
                c.flags &= ~kPresentPending;
            }
        }
        // Settle the dots since the last event (only a console that faulted
        // stops between events).
        if (static_cast<std::uint32_t>(cpu.left) != uni(c.r32(reg::kHorizon))) {
            c.w32(reg::kFrames, c.r32(reg::kFrames) + c.settle(c.r32(reg::kHorizon) - static_cast<std::uint32_t>(cpu.left), true));
            if (c.flags & kPresentPending) C::capture(c.s, env, c.regs_base, lane, 64);
        }
        flags = c.flags;
        frames = c.r32(reg::kFrames);
        // Whether the first consoles took the general path too often.
        if (blockIdx.x < kGeneralSlots && wave == 0 && lane == 0) {
            KState* k = reload(c.s);
            const GeneralLimit limit{k->general_idle, k->general_busy};
            k->choice->over[blockIdx.x] = over_limit(limit, general, jumps, frameskip, kFrameDots) ? 1u : 0u;
        }
    }
    __syncthreads();

    // RAM rows back to HBM.
    std::uint8_t* ram = reload(c.s)->ram;
    if (W >= 4) {
        for (std::uint32_t q = 0; q < W && env0 + q < P; q += 4) {
            for (std::uint32_t row = tid; row < kRamBytes; row += T) {
                const std::uint8_t* at = lds + kWaveRam + q * kRamBytes + row;
                *reinterpret_cast<std::uint32_t*>(ram + static_cast<std::size_t>(row) * P + env0 + q) =
                    at[0] | (at[kRamBytes] << 8) | (at[2 * kRamBytes] << 16) |
                    (static_cast<std::uint32_t>(at[3 * kRamBytes]) << 24);
            }
        }
    } else {
        for (std::uint32_t q = 0; q < W; ++q)
            for (std::uint32_t row = tid; row < kRamBytes; row += T)
                ram[static_cast<std::size_t>(row) * P + env0 + q] = lds[kWaveRam + q * kRamBytes + row];
    }
    if (!mine || lane != 0) return;
    KState& es = *reload(c.s);
    const std::uint32_t fd = c.r32(reg::kFrameDot);
    es.pc[env] = static_cast<std::uint16_t>(cpu.pc);
    es.a[env] = static_cast<std::uint8_t>(cpu.a);
    es.x[env] = static_cast<std::uint8_t>(cpu.x);
    es.y[env] = static_cast<std::uint8_t>(cpu.y);
    es.sp[env] = static_cast<std::uint8_t>(cpu.sp);
    es.p[env] = static_cast<std::uint8_t>(cpu.p);
    // Every CPU cycle is 3 PPU dots.
    const std::uint64_t advanced = static_cast<std::uint64_t>(frames) * kFrameDots + fd - fd0;
    es.cycles[env] += advanced / 3;
    es.frame[env] += frames;
    es.frame_dot[env] = fd;
    es.nmi_pending[env] = static_cast<std::uint8_t>((flags & kNmiPending) ? 1 : 0);
    es.status[env] = static_cast<std::uint8_t>(c.status());
    es.ctrl[env] = static_cast<std::uint8_t>(c.r8(reg::kCtrl));
    es.mask[env] = static_cast<std::uint8_t>(c.r8(reg::kMask));
    es.oam_addr[env] = static_cast<std::uint8_t>(c.r8(reg::kOamAddr));
    es.open_bus[env] = static_cast<std::uint8_t>(c.open_bus());
    es.read_buffer[env] = static_cast<std::uint8_t>(c.r8(reg::kReadBuffer));
    es.v[env] = static_cast<std::uint16_t>(c.r16(reg::kV));
    es.t[env] = static_cast<std::uint16_t>(c.r16(reg::kT));
    es.fine_x[env] = static_cast<std::uint8_t>(c.r8(reg::kFineX));
    es.w[env] = static_cast<std::uint8_t>((flags & kWToggle) ? 1 : 0);
    es.scroll_x[env] = static_cast<std::uint8_t>(c.r8(reg::kScrollX));
    es.scroll_y[env] = static_cast<std::uint8_t>(c.r8(reg::kScrollY));
    es.c1_buttons[env] = static_cast<std::uint8_t>(c.buttons());
    es.c1_shift[env] = static_cast<std::uint8_t>(c.c1_shift());
    es.c1_count[env] = static_cast<std::uint8_t>(c.c1_count());
    es.strobe[env] = static_cast<std::uint8_t>((flags & kStrobeBit) ? 1 : 0);
    es.c2_count[env] = static_cast<std::uint8_t>(c.c2_count());
    const bool fault = (flags & kFault) != 0;
    es.fault[env] = static_cast<std::uint8_t>(fault ? 1 : 0);
    float reward = 0.0f;
    std::uint32_t done = 1;
    if (!fault)
        reward_apply(es, env, [&](std::uint32_t a) -> std::uint32_t { return lds[base + (a & 0x7FF)]; }, &reward, &done);
    es.rewards[env] = reward;
    es.done[env] = static_cast<std::uint8_t>(done);
}

}  // namespace

// Waves per workgroup: as few as keep the batch within one workgroup per CU,
// so that every CU has its share; more than 16 a CU become two workgroups.
// Of those, 12 waves where the chip's 512 resident workgroups then take no
// round more than with 16, as six waves per SIMD end sooner than eight and a
// few workgroups left for a last round run longer beside a full one.  ms per
// step with 16 -> 12 waves: one round, 4,097 consoles 3.34 -> 3.03, 6,144 3.35
// -> 2.99 (frame-skip 1 0.97 -> 0.81, a game that idles 1.18 -> 1.02); a second
// round of at most one workgroup per CU, 8,200 6.23 -> 5.64, 9,200 6.43 ->
// 5.40 (beyond it 9,400 6.08 -> 6.00, but 1.53 -> 1.66 at frame-skip 1); a
// third, 16,400 9.10 -> 8.64, 18,200 8.88 -> 8.60, but 2.32 -> 2.39 at
// frame-skip 1, where loads and stores weigh more: only from frame-skip 4.
hipError_t NESLE_WAVE_LAUNCH(const DeviceState& s, std::uint32_t frameskip, hipStream_t stream) {
    constexpr std::uint32_t kCus = 256, kResident = 2 * kCus, kFewer = 12;
    std::uint32_t waves = (s.n + kCus - 1) / kCus;
    if (waves > 2) waves = (waves + 3) & ~3u;
    if (waves > kWaveMaxWaves) {
        const std::uint32_t round = kResident * kWaveMaxWaves, fewer = (s.n + kFewer - 1) / kFewer;
        const bool pays = s.n <= round ? fewer <= kResident
                          : s.n <= 2 * round ? fewer <= kResident + kCus
                                             : fewer <= 3 * kResident && frameskip >= 4;
        waves = pays ? kFewer : kWaveMaxWaves;
    }
    NESLE_WAVE_KERNEL<<<dim3((s.n + waves - 1) / waves), dim3(64 * waves), 0, stream>>>(s, frameskip);
    return hipGetLastError();
}

}  // namespace nesle
