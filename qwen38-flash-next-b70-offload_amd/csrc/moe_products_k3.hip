// The grouped experts' products at 3 bits.
#include "moe_products.cuh"

namespace exl3 {
template void launch_products<3>(const GroupedArgs& a, bool y32, hipStream_t s);
}  // namespace exl3
