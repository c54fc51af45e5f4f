// Instantiates the Cauchy-product matmul kernels for one type.
#include "cauchy_matmul.inl"

namespace pt {
template int launch_cauchy<float>(const CauchyArgs&);
template int launch_order_sum<float>(const OrderSumArgs&);
}  // namespace pt
