// Elementwise activations along complex directions: the real series at the K + 1 interpolation nodes and
// their combination (complex_planes.hip), in one streaming pass with everything between in registers.
//
// Bound by memory: base and K complex planes are read once and written once. As separate passes (the
// variants of every node, an activation per node, the combination) 7 + 12, 32 and 18 real planes were
// moved at K = 3 where 14 are needed. 1024 x 3072 complex64, degree 3, tanh GELU: 47 us (3.7 TB/s), the block
// of a decoder it belongs to 1734 -> 1620 us.
#include "activation_series.inl"

namespace pt {

template <typename T>
struct ComplexActArgs {
  const T* x0;
  T* y0;
  const T* src[PT_MAX_DEGREE];   // interleaved (re, im) planes of orders 1..K
  T* dst[PT_MAX_DEGREE];
  T node[PT_MAX_DEGREE + 1], wre[PT_MAX_DEGREE + 1], wim[PT_MAX_DEGREE + 1];
};

// One element: p holds (re, im) of orders 1..K at p[k - 1][at], [at + 1], in and out.
template <typename T, int K, int N>
__device__ __forceinline__ T complex_activation_element(int kind, const ComplexActArgs<T>& a, T x0, T (&p)[K][N], int at) {
  T re[K], im[K], y0 = T(0);
#pragma unroll
  for (int k = 0; k < K; ++k) re[k] = im[k] = T(0);
#pragma unroll 1   // (a body of K + 1 series for every kind would not fit the instruction cache)
  for (int m = 0; m <= K; ++m) {
    T u[K + 1], out[K + 1];
    u[0] = x0;
#pragma unroll
    for (int k = 1; k <= K; ++k) u[k] = p[k - 1][at] + a.node[m] * p[k - 1][at + 1];
    activation_element<T, K, false>(kind, u, u, out);
    y0 = out[0];   // the same at every node
#pragma unroll
    for (int k = 1; k <= K; ++k) {
      re[k - 1] += a.wre[m] * out[k];
      im[k - 1] += a.wim[m] * out[k];
    }
  }
#pragma unroll
  for (int k = 0; k < K; ++k) {
    p[k][at] = re[k];
    p[k][at + 1] = im[k];
  }
  return y0;
}

// vec: every pointer 16-byte aligned; a thread then takes one 16-byte vector of base values and two of
// every plane.
template <typename T, int K>
__global__ __launch_bounds__(kActThreads) void complex_activation_kernel(int kind, ComplexActArgs<T> a, int64_t numel,
                                                                         bool vec) {
  constexpr int V = 16 / static_cast<int>(sizeof(T));
  const int64_t stride = static_cast<int64_t>(gridDim.x) * kActThreads;
  const int64_t first = static_cast<int64_t>(blockIdx.x) * kActThreads + threadIdx.x;
  const int64_t groups = vec ? numel / V : 0;
  for (int64_t g = first; g < groups; g += stride) {
    Vec<T, V> x0 = load_vec_nt<T, V>(a.x0 + V * g);
    T p[K][2 * V];
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const Vec<T, V> c0 = load_vec_nt<T, V>(a.src[k] + 2 * V * g), c1 = load_vec_nt<T, V>(a.src[k] + 2 * V * g + V);
#pragma unroll
      for (int e = 0; e < V; ++e) {
        p[k][e] = c0.v[e];
        p[k][V + e] = c1.v[e];
      }
    }
#pragma unroll
    for (int e = 0; e < V; ++e) x0.v[e] = complex_activation_element<T, K, 2 * V>(kind, a, x0.v[e], p, 2 * e);
    store_vec_nt<T, V>(a.y0 + V * g, x0);
#pragma unroll
    for (int k = 0; k < K; ++k) {
      Vec<T, V> c0, c1;
#pragma unroll
      for (int e = 0; e < V; ++e) {
        c0.v[e] = p[k][e];
        c1.v[e] = p[k][V + e];
      }
      store_vec_nt<T, V>(a.dst[k] + 2 * V * g, c0);
      store_vec_nt<T, V>(a.dst[k] + 2 * V * g + V, c1);
    }
  }
  for (int64_t i = groups * V + first; i < numel; i += stride) {
    T p[K][2];
#pragma unroll
    for (int k = 0; k < K; ++k) {
      p[k][0] = a.src[k][2 * i];
      p[k][1] = a.src[k][2 * i + 1];
    }
    a.y0[i] = complex_activation_element<T, K, 2>(kind, a, a.x0[i], p, 0);
#pragma unroll
    for (int k = 0; k < K; ++k) {
      a.dst[k][2 * i] = p[k][0];
      a.dst[k][2 * i + 1] = p[k][1];
    }
  }
}

template <typename T, int K>
static int launch_complex_activation_k(int kind, const ComplexActArgs<T>& a, int64_t numel, hipStream_t stream) {
  constexpr int V = 16 / static_cast<int>(sizeof(T));
  bool vec = pt_host::aligned16(a.x0) && pt_host::aligned16(a.y0);
  for (int k = 0; k < K; ++k) vec = vec && pt_host::aligned16(a.src[k]) && pt_host::aligned16(a.dst[k]);
  const int64_t work = vec ? numel / V + numel % V : numel;
  const int64_t blocks = std::max<int64_t>(1, std::min<int64_t>((work + kActThreads - 1) / kActThreads, kActMaxBlocks));
  complex_activation_kernel<T, K><<<dim3(static_cast<unsigned>(blocks)), dim3(kActThreads), 0, stream>>>(kind, a, numel, vec);
  PT_LAUNCH_CHECK();
  return PT_OK;
}

template <typename T>
static int launch_complex_activation(int degree, int kind, const void* x0, const void* const* x, void* y0, void* const* y,
                                     const double* nodes, const double* wre, const double* wim, int64_t numel,
                                     hipStream_t stream) {
  ComplexActArgs<T> a{};
  a.x0 = static_cast<const T*>(x0);
  a.y0 = static_cast<T*>(y0);
  for (int k = 0; k < degree; ++k) {
    a.src[k] = static_cast<const T*>(x[k]);
    a.dst[k] = static_cast<T*>(y[k]);
  }
  for (int m = 0; m <= degree; ++m) {
    a.node[m] = static_cast<T>(nodes[m]);
    a.wre[m] = static_cast<T>(wre[m]);
    a.wim[m] = static_cast<T>(wim[m]);
  }
  switch (degree) {
    case 1: return launch_complex_activation_k<T, 1>(kind, a, numel, stream);
    case 2: return launch_complex_activation_k<T, 2>(kind, a, numel, stream);
    case 3: return launch_complex_activation_k<T, 3>(kind, a, numel, stream);
    case 4: return launch_complex_activation_k<T, 4>(kind, a, numel, stream);
    case 5: return launch_complex_activation_k<T, 5>(kind, a, numel, stream);
    case 6: return launch_complex_activation_k<T, 6>(kind, a, numel, stream);
    case 7: return launch_complex_activation_k<T, 7>(kind, a, numel, stream);
    default: return launch_complex_activation_k<T, 8>(kind, a, numel, stream);
  }
}

}  // namespace pt

extern "C" int pt_complex_activation_fwd(int dtype, int degree, int kind, const void* x0, const void* const* x, void* y0,
                                         void* const* y, const double* nodes, const double* wre, const double* wim,
                                         int64_t numel, void* stream) {
  pt_host::clear_error();
  PT_REQUIRE(degree >= 1 && degree <= PT_MAX_DEGREE, PT_UNSUPPORTED, "complex activation: degree must be in 1..8");
  PT_REQUIRE(dtype == PT_FLOAT32 || dtype == PT_FLOAT64, PT_UNSUPPORTED, "complex activation: float32 or float64");
  PT_REQUIRE(kind >= PT_ACT_GELU && kind <= PT_ACT_RSQRT, PT_UNSUPPORTED, "complex activation: unknown activation kind");
  PT_REQUIRE(numel >= 0, PT_INVALID_ARGUMENT, "complex activation: numel must be >= 0");
  PT_REQUIRE(x != nullptr && y != nullptr && nodes != nullptr && wre != nullptr && wim != nullptr, PT_INVALID_ARGUMENT,
             "complex activation: pointer arrays, nodes and weights are required");
  if (numel == 0) return PT_OK;
  PT_REQUIRE(x0 != nullptr && y0 != nullptr, PT_INVALID_ARGUMENT, "complex activation: null coefficient pointer");
  for (int k = 0; k < degree; ++k)
    PT_REQUIRE(x[k] != nullptr && y[k] != nullptr, PT_INVALID_ARGUMENT, "complex activation: null coefficient pointer");
  const auto s = static_cast<hipStream_t>(stream);
  if (dtype == PT_FLOAT32)
    return pt::launch_complex_activation<float>(degree, kind, x0, x, y0, y, nodes, wre, wim, numel, s);
  return pt::launch_complex_activation<double>(degree, kind, x0, x, y0, y, nodes, wre, wim, numel, s);
}
