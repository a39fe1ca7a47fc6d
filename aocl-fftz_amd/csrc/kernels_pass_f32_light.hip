// Instantiation unit: single-size pass kernels with the radices of kRadLight,
// complex64; 256- or 1024-thread bound.
#include "kernels_body.h"

namespace fftz {

const void* kernel_symbol_pass_f32_light(KernelKind kind, bool nt, int maxt)
{
    return sym_t<float, kRadLight>(kind, nt, maxt);
}

}  // namespace fftz
