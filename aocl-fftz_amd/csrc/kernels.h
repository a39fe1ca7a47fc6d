// Kernel symbols exported from the kernel units to the host planner.
#pragma once

#include "pass.h"

namespace fftz {

enum class KernelKind { Pass, Real, RealWide, Bluestein };

// Radices a generic kernel carries.  The widest butterfly it carries sets the
// registers, and with them the wavefronts, of every launch; wavefronts per SIMD
// of the plain pass in complex64 / complex128: kRadAll 4 / 3, kRadLight 5 / 3,
// kRadTo8 - / 4; of Bluestein: kRadAll 5 / 2, kRadLight 5 / 3, kRadTo8 - / 4.
enum RadixSet : int {
    kRadPow2 = 0,   // 2, 4, 8, 16
    kRadAll = 1,    // 2 .. 13, 16
    kRadLight = 2,  // 2 .. 12; no real passes
    kRadTo8 = 3,    // 2 .. 8, complex128 only; mirrored pairs of radix 2 .. 6
};

constexpr bool rad_in_set(int set, int r)
{
    return set == kRadPow2    ? (r & (r - 1)) == 0
           : set == kRadLight ? r <= 12
           : set == kRadTo8   ? r <= 8
                              : true;
}

// Radices of the stage that holds mirrored butterfly pairs (two butterflies'
// registers at once).
constexpr bool rad_in_pairs(int set, int r) { return r <= (set == kRadTo8 ? 6 : 10) && rad_in_set(set, r); }

// Device function symbol for hipLaunchKernel / hipFuncSetAttribute; nullptr
// where there is no such kernel.  prec_bytes: 4 (complex64) or 8 (complex128).
// rad: a RadixSet.  nt: the variant whose complex results bypass the L2's
// write-back (kNtStore).  maxt: block-size bound of the variant, 256 or more
// (then 1024 threads in complex64, 512 in complex128); the 256 variants get a
// larger VGPR budget.  Real: passes with a real side (kRealFlags); RealWide:
// real-packed ones whose pair stage (last for R2C, first for C2R) has a radix
// above 10: 11 or 13 where the length has no other, any in a tuned order.
const void* kernel_symbol(KernelKind kind, int prec_bytes, int rad, bool nt, int maxt);

// Uneven-batch persistent kernel (k_batch) of a tile class (0 small: 256
// threads, 1 medium: 512, 2 large: 1024 in complex64, 512 in complex128), and the
// counter reset kernel launched before it.  nt: results bypass the L2's
// write-back (those of the medium and large class always do).
const void* kernel_symbol_batch(int prec_bytes, int cls, bool nt);
const void* kernel_symbol_reset();

// Instantiation units behind kernel_symbol / kernel_symbol_batch (one
// translation unit each, compiled in parallel).
const void* kernel_symbol_pass_f32_mixed(KernelKind kind, bool nt, int maxt);
const void* kernel_symbol_pass_f32_pow2(KernelKind kind, bool nt, int maxt);
const void* kernel_symbol_pass_f64_mixed(KernelKind kind, bool nt, int maxt);
const void* kernel_symbol_pass_f64_pow2(KernelKind kind, bool nt, int maxt);
const void* kernel_symbol_pass_f32_light(KernelKind kind, bool nt, int maxt);
const void* kernel_symbol_pass_f64_light(KernelKind kind, bool nt, int maxt);
const void* kernel_symbol_pass_f64_to8(KernelKind kind, bool nt, int maxt);
const void* kernel_symbol_batch_f32_small(bool nt);
const void* kernel_symbol_batch_f32_medium();
const void* kernel_symbol_batch_f32_large();
const void* kernel_symbol_batch_f64_small(bool nt);
const void* kernel_symbol_batch_f64_medium();
const void* kernel_symbol_batch_f64_large();

// Fixed-length pass kernel for power-of-two L in [64, 4096] (radix plan 16s
// then remainder, 16 elements per thread), block <= maxt (256, or 512 for
// L >= 256); nullptr otherwise.  split (complex64 L = 512, complex128 L = 256):
// stage exchanges of the real and the imaginary parts in turn, through half
// the LDS.  nt: results bypass the L2's write-back.
const void* kernel_symbol_fixed(int prec_bytes, int L, int maxt, bool split, bool nt);

// Matrix-core pass (kernels_mfma.hip) for complex64, L = 256 or 4096, with
// operand precision `mode` (MfmaMode) and nb (2 or 4) column blocks per
// wavefront (block = 1024 / nb threads); nullptr for other arguments.
// Kernel arguments: (PassDesc, const float* fragments).
const void* kernel_symbol_mfma(int mode, int L, int nb);

}  // namespace fftz
