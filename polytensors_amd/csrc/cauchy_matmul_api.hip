// C ABI of the Cauchy-product matmul kernels.
#include "cauchy_matmul.h"

#include <algorithm>

namespace pt {

// Row-padded copies, blockIdx.y the matrix: one 16-byte vector of the destination per thread and step,
// read at any element's address; the vector across a row's end by elements. Bound by the copy: the ten
// orders of 4 x 511 x 1023 and 4 x 1023 x 769 bfloat16 operands (34 MB read, 34 written) take 23 us in
// two launches, where a padded copy and a fill of each order took 130.
template <typename E>
__global__ __launch_bounds__(256) void pack_rows_kernel(CPtrs<E> src, MPtrs<E> dst, int64_t rows, int64_t cols,
                                                        int64_t vecs /* of a destination row */) {
  constexpr int V = 16 / static_cast<int>(sizeof(E));
  const E* __restrict__ from = src.p[blockIdx.y];
  E* __restrict__ to = dst.p[blockIdx.y];
  const int64_t step = static_cast<int64_t>(gridDim.x) * 256;
  int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  int64_t r = i / vecs, v = i % vecs;
  const int64_t step_r = step / vecs, step_v = step % vecs;
  while (r < rows) {
    Vec<E, V> x;
    const E* p = from + r * cols + v * V;
    if (v * V + V <= cols) {
      __builtin_memcpy(&x, p, sizeof(x));
    } else {
#pragma unroll
      for (int e = 0; e < V; ++e) x.v[e] = v * V + e < cols ? p[e] : E(0);
    }
    store_vec<E, V>(to + (r * vecs + v) * V, x);
    r += step_r;
    v += step_v;
    if (v >= vecs) {
      v -= vecs;
      ++r;
    }
  }
}

template <typename E>
static int launch_pack(int count, const void* const* src, void* const* dst, int64_t rows, int64_t cols, int64_t dst_cols,
                       hipStream_t stream) {
  CPtrs<E> from{};
  MPtrs<E> to{};
  for (int i = 0; i < count; ++i) {
    from.p[i] = static_cast<const E*>(src[i]);
    to.p[i] = static_cast<E*>(dst[i]);
  }
  const int64_t vecs = dst_cols / (16 / static_cast<int64_t>(sizeof(E)));
  const int64_t blocks = std::min<int64_t>((rows * vecs + 255) / 256, 2048);
  pack_rows_kernel<E><<<dim3(static_cast<unsigned>(blocks), static_cast<unsigned>(count)), dim3(256), 0, stream>>>(
      from, to, rows, cols, vecs);
  PT_LAUNCH_CHECK();
  return PT_OK;
}

int launch_pack_rows(int elem_bytes, int count, const void* const* src, void* const* dst, int64_t rows, int64_t cols,
                     int64_t dst_cols, hipStream_t stream) {
  if (elem_bytes == 2) return launch_pack<uint16_t>(count, src, dst, rows, cols, dst_cols, stream);
  if (elem_bytes == 4) return launch_pack<uint32_t>(count, src, dst, rows, cols, dst_cols, stream);
  return launch_pack<uint64_t>(count, src, dst, rows, cols, dst_cols, stream);
}

}  // namespace pt

extern "C" {

int pt_cauchy_matmul(int dtype, int degree, const void* const* a, int a_orders,
                     const void* const* b, int b_orders, void* const* c, int64_t batch, int64_t m,
                     int64_t n, int64_t k, int64_t a_batch_stride, int64_t b_batch_stride,
                     int trans_b, void* stream) {
  return pt_cauchy_matmul_strided(dtype, degree, a, a_orders, b, b_orders, c, batch, m, n, k, k, trans_b ? k : n,
                                  a_batch_stride, b_batch_stride, trans_b, nullptr, stream);
}

int pt_cauchy_matmul_strided(int dtype, int degree, const void* const* a, int a_orders, const void* const* b,
                             int b_orders, void* const* c, int64_t batch, int64_t m, int64_t n, int64_t k, int64_t lda,
                             int64_t ldb, int64_t a_batch_stride, int64_t b_batch_stride, int trans_b, const void* bias,
                             void* stream) {
  pt_host::clear_error();
  PT_REQUIRE(degree >= 0 && degree <= PT_MAX_DEGREE, PT_UNSUPPORTED,
             "Cauchy matmul: degree must be in 0..8");
  PT_REQUIRE(dtype == PT_FLOAT32 || dtype == PT_FLOAT64 || dtype == PT_BFLOAT16 || dtype == PT_FLOAT16,
             PT_UNSUPPORTED, "Cauchy matmul: float32, float64, bfloat16 or float16");
  PT_REQUIRE(a != nullptr && b != nullptr && c != nullptr, PT_INVALID_ARGUMENT,
             "Cauchy matmul: a, b and c pointer arrays are required");
  PT_REQUIRE(a_orders == 1 || a_orders == degree + 1, PT_INVALID_ARGUMENT,
             "Cauchy matmul: a_orders must be 1 or degree+1");
  PT_REQUIRE(b_orders == 1 || b_orders == degree + 1, PT_INVALID_ARGUMENT,
             "Cauchy matmul: b_orders must be 1 or degree+1");
  PT_REQUIRE(batch >= 0 && m >= 0 && n >= 0 && k >= 0, PT_INVALID_ARGUMENT,
             "Cauchy matmul: negative size");
  PT_REQUIRE(a_batch_stride >= 0 && b_batch_stride >= 0, PT_INVALID_ARGUMENT,
             "Cauchy matmul: negative batch stride");
  PT_REQUIRE(lda >= k && ldb >= (trans_b ? k : n), PT_INVALID_ARGUMENT,
             "Cauchy matmul: a row stride below the row length");
  PT_REQUIRE(lda <= INT32_MAX && ldb <= INT32_MAX, PT_UNSUPPORTED,
             "Cauchy matmul: a row stride beyond 2^31 - 1 elements");   // (the kernels take 32-bit strides)
  PT_REQUIRE(m <= INT32_MAX && n <= INT32_MAX && k <= INT32_MAX && batch <= 65535 &&
                 (m + 31) / 32 <= 65535,
             PT_UNSUPPORTED, "Cauchy matmul: sizes beyond the launch grid");
  for (int o = 0; o < a_orders; ++o)
    PT_REQUIRE(a[o] != nullptr, PT_INVALID_ARGUMENT, "Cauchy matmul: null A coefficient");
  for (int o = 0; o < b_orders; ++o)
    PT_REQUIRE(b[o] != nullptr, PT_INVALID_ARGUMENT, "Cauchy matmul: null B coefficient");
  for (int o = 0; o <= degree; ++o)
    PT_REQUIRE(c[o] != nullptr, PT_INVALID_ARGUMENT, "Cauchy matmul: null C coefficient");
  if (batch == 0 || m == 0 || n == 0) return PT_OK;
  pt::CauchyArgs args{degree, a, a_orders, b, b_orders, c, batch, m, n, k, lda, ldb,
                      a_batch_stride, b_batch_stride, trans_b != 0, bias, static_cast<hipStream_t>(stream)};
  switch (dtype) {
    case PT_FLOAT32: return pt::launch_cauchy<float>(args);
    case PT_FLOAT64: return pt::launch_cauchy<double>(args);
    case PT_BFLOAT16: return pt::launch_cauchy_half<pt::bf16>(args);
    default: return pt::launch_cauchy_half<_Float16>(args);
  }
}

int pt_pack_rows(int elem_bytes, int count, const void* const* src, void* const* dst, int64_t rows, int64_t cols,
                 int64_t dst_cols, void* stream) {
  pt_host::clear_error();
  PT_REQUIRE(elem_bytes == 2 || elem_bytes == 4 || elem_bytes == 8, PT_INVALID_ARGUMENT,
             "pack rows: elements of 2, 4 or 8 bytes");
  PT_REQUIRE(count >= 1 && count <= PT_MAX_DEGREE + 1, PT_INVALID_ARGUMENT, "pack rows: count must be in 1..9");
  PT_REQUIRE(rows >= 0 && cols >= 0 && dst_cols >= cols && dst_cols * elem_bytes % 16 == 0, PT_INVALID_ARGUMENT,
             "pack rows: dst_cols must hold cols in whole 16-byte vectors");
  PT_REQUIRE(src != nullptr && dst != nullptr, PT_INVALID_ARGUMENT, "pack rows: src and dst are required");
  if (rows == 0 || dst_cols == 0) return PT_OK;
  for (int i = 0; i < count; ++i)
    PT_REQUIRE((src[i] != nullptr || cols == 0) && dst[i] != nullptr && pt_host::aligned16(dst[i]), PT_INVALID_ARGUMENT,
               "pack rows: null or unaligned matrix");
  return pt::launch_pack_rows(elem_bytes, count, src, dst, rows, cols, dst_cols, static_cast<hipStream_t>(stream));
}

int pt_matmul_order_sum(int dtype, int terms, const void* const* a, const void* const* b, void* c, int64_t batch,
                        int64_t m, int64_t n, int64_t k, int64_t lda, int64_t ldb, int64_t a_batch_stride,
                        int64_t b_batch_stride, int trans_a, int trans_b, void* stream) {
  pt_host::clear_error();
  PT_REQUIRE(terms >= 1 && terms <= PT_MAX_DEGREE + 1, PT_INVALID_ARGUMENT, "matmul order sum: terms must be in 1..9");
  PT_REQUIRE(dtype == PT_FLOAT32 || dtype == PT_BFLOAT16 || dtype == PT_FLOAT16, PT_UNSUPPORTED,
             "matmul order sum: float32, bfloat16 or float16");
  PT_REQUIRE(!(trans_a && trans_b), PT_UNSUPPORTED, "matmul order sum: trans_a needs trans_b = 0");
  PT_REQUIRE(batch >= 0 && m >= 0 && n >= 0 && k >= 0 && a_batch_stride >= 0 && b_batch_stride >= 0, PT_INVALID_ARGUMENT,
             "matmul order sum: negative size or batch stride");
  PT_REQUIRE(lda >= (trans_a ? m : k) && ldb >= (trans_b ? k : n), PT_INVALID_ARGUMENT,
             "matmul order sum: a row stride below the row length");
  if (batch == 0 || m == 0 || n == 0) return PT_OK;
  PT_REQUIRE(a != nullptr && b != nullptr && c != nullptr, PT_INVALID_ARGUMENT,
             "matmul order sum: a, b and c are required");
  for (int s = 0; s < terms; ++s)
    PT_REQUIRE((a[s] != nullptr && b[s] != nullptr) || k == 0, PT_INVALID_ARGUMENT, "matmul order sum: null operand");
  pt::OrderSumArgs args{terms, a, b, c, batch, m, n, k, lda, ldb, a_batch_stride, b_batch_stride,
                        trans_a != 0, trans_b != 0, static_cast<hipStream_t>(stream)};
  switch (dtype) {
    case PT_FLOAT32: return pt::launch_order_sum<float>(args);
    case PT_BFLOAT16: return pt::launch_order_sum<pt::bf16>(args);
    default: return pt::launch_order_sum<_Float16>(args);
  }
}

}  // extern "C"
