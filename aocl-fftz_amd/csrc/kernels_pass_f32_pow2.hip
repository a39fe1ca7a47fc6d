// Instantiation unit: single-size pass, real and Bluestein kernels with radices 2, 4, 8, 16,
// complex64; 256- or 1024-thread bound.
#include "kernels_body.h"

namespace fftz {

const void* kernel_symbol_pass_f32_pow2(KernelKind kind, bool nt, int maxt)
{
    return sym_t<float, kRadPow2>(kind, nt, maxt);
}

}  // namespace fftz
