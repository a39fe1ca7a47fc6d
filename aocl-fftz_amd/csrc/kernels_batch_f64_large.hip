// Instantiation unit: uneven-batch persistent kernel, large class: 512 threads, complex128.
// (One kernel per unit: the units compile in parallel.)
#include "kernels_body.h"

namespace fftz {

const void* kernel_symbol_batch_f64_large() { return (const void*)&k_batch<double, 512, true>; }

}  // namespace fftz
