// The grouped experts' products at 4 bits.
#include "moe_products.cuh"

namespace exl3 {
template void launch_products<4>(const GroupedArgs& a, bool y32, hipStream_t s);
}  // namespace exl3
