// Instantiates the 16-bit Cauchy-product matmul kernels for one type.
#include "cauchy_matmul_half.inl"

namespace pt {
template int launch_cauchy_half<_Float16>(const CauchyArgs&);
template int launch_order_sum<_Float16>(const OrderSumArgs&);
}  // namespace pt
