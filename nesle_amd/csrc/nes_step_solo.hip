// nes_step_solo.hip -- the one-console-per-wave step kernel for few waves per
// SIMD (up to 4,096 consoles), built from nes_step_wave.hip with the form of
// its assembly that is quickest for a wave of its own (SOLO in nes_wave.h).
#define NESLE_WAVE_SOLO "1"
#define NESLE_WAVE_KERNEL solo_kernel
#define NESLE_WAVE_LAUNCH launch_step_solo
#include "nes_step_wave.hip"
