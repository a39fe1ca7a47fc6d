// Instantiation unit: uneven-batch persistent kernel, small class: 256 threads, complex128.
// (One kernel per unit: the units compile in parallel.)
#include "kernels_body.h"

namespace fftz {

const void* kernel_symbol_batch_f64_small() { return (const void*)&k_batch<double, 256>; }

}  // namespace fftz
