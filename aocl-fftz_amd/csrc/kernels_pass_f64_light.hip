// Instantiation unit: single-size pass kernels with the radices of kRadLight,
// complex128; 256- or 512-thread bound.
#include "kernels_body.h"

namespace fftz {

const void* kernel_symbol_pass_f64_light(KernelKind kind, bool nt, int maxt)
{
    return sym_t<double, kRadLight>(kind, nt, maxt);
}

}  // namespace fftz
