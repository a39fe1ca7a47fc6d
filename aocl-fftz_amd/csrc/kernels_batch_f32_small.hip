// Instantiation unit: uneven-batch persistent kernel, small class: 256 threads, complex64.
// (One class per unit: the units compile in parallel.)
#include "kernels_body.h"

namespace fftz {

const void* kernel_symbol_batch_f32_small(bool nt)
{
    return nt ? (const void*)&k_batch<float, 256, true> : (const void*)&k_batch<float, 256, false>;
}

}  // namespace fftz
