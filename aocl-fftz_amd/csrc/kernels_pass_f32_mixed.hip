// Instantiation unit: single-size pass, real and Bluestein kernels with every radix (2-13),
// complex64; 256- or 1024-thread bound.
#include "kernels_body.h"

namespace fftz {

const void* kernel_symbol_pass_f32_mixed(KernelKind kind, bool nt, int maxt)
{
    return sym_t<float, kRadAll>(kind, nt, maxt);
}

}  // namespace fftz
