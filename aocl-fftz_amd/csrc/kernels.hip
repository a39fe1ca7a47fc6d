// Launch table of the LDS pass kernels: precision x radix set x block
// limit.  The kernels themselves are instantiated in
// kernels_pass_{f32,f64}_{mixed,pow2,light}.hip, kernels_pass_f64_to8.hip and
// kernels_batch_{f32,f64}_{small,medium,large}.hip (one translation unit
// each, so they compile in parallel) from kernels_body.h.
#include <hip/hip_runtime.h>

#include "kernels.h"

namespace fftz {

// Clears the uneven batch's work-queue counters (a kernel rather than a
// memset node, so the launch sequence can be captured in a graph).
__global__ void k_reset_counters(unsigned* c, int n)
{
    if ((int)threadIdx.x < n) c[threadIdx.x] = 0u;
}

const void* kernel_symbol(KernelKind kind, int prec_bytes, int rad, bool nt, int maxt)
{
    if (prec_bytes == 4) switch (rad) {
            case kRadPow2: return kernel_symbol_pass_f32_pow2(kind, nt, maxt);
            case kRadAll: return kernel_symbol_pass_f32_mixed(kind, nt, maxt);
            case kRadLight: return kernel_symbol_pass_f32_light(kind, nt, maxt);
            default: return nullptr;
        }
    switch (rad) {
        case kRadPow2: return kernel_symbol_pass_f64_pow2(kind, nt, maxt);
        case kRadAll: return kernel_symbol_pass_f64_mixed(kind, nt, maxt);
        case kRadLight: return kernel_symbol_pass_f64_light(kind, nt, maxt);
        case kRadTo8: return kernel_symbol_pass_f64_to8(kind, nt, maxt);
        default: return nullptr;
    }
}

const void* kernel_symbol_batch(int prec_bytes, int cls, bool nt)
{
    if (cls == 0) return prec_bytes == 4 ? kernel_symbol_batch_f32_small(nt) : kernel_symbol_batch_f64_small(nt);
    if (cls == 1) return prec_bytes == 4 ? kernel_symbol_batch_f32_medium() : kernel_symbol_batch_f64_medium();
    return prec_bytes == 4 ? kernel_symbol_batch_f32_large() : kernel_symbol_batch_f64_large();
}

const void* kernel_symbol_reset() { return (const void*)&k_reset_counters; }

}  // namespace fftz
