// Launch interface of the Cauchy-product matmul kernels (definitions in cauchy_matmul.inl).
#pragma once

#include "pt_common.h"

namespace pt {

struct CauchyArgs {
  int degree;
  const void* const* a;
  int a_orders;
  const void* const* b;
  int b_orders;
  void* const* c;
  int64_t batch, m, n, k;
  int64_t lda, ldb;   // row strides; zeros from k to the next 16-byte vector where rows run along k
  int64_t a_bs, b_bs;
  bool trans_b;
  const void* bias;   // null, or n values added to every row of order 0
  hipStream_t stream;
  int64_t rows_b() const { return trans_b ? n : k; }
  int64_t width_b() const { return trans_b ? k : n; }
};

template <typename T>
int launch_cauchy(const CauchyArgs& a);

// C = sum_s op(A_s) op(B_s) over `terms` pairs (order_gemm.inl).
struct OrderSumArgs {
  int terms;
  const void* const* a;
  const void* const* b;
  void* c;
  int64_t batch, m, n, k, lda, ldb, a_bs, b_bs;
  bool trans_a, trans_b;
  hipStream_t stream;
};

// Copies of `count` [rows, cols] matrices with rows padded by zeros to dst_cols (cauchy_matmul_api.hip).
int launch_pack_rows(int elem_bytes, int count, const void* const* src, void* const* dst, int64_t rows, int64_t cols,
                     int64_t dst_cols, hipStream_t stream);

template <typename T>
int launch_order_sum(const OrderSumArgs& a);   // float, bf16, _Float16

// bfloat16 / float16 operands on the 16x16x32 MFMAs (cauchy_matmul_half.inl); T = bf16 or _Float16.
template <typename T>
int launch_cauchy_half(const CauchyArgs& a);

}  // namespace pt
