// Instantiation unit: single-size pass, real and Bluestein kernels with every radix (2-13),
// complex128; 256- or 512-thread bound.
#include "kernels_body.h"

namespace fftz {

const void* kernel_symbol_pass_f64_mixed(KernelKind kind, bool nt, int maxt)
{
    return sym_t<double, kRadAll>(kind, nt, maxt);
}

}  // namespace fftz
