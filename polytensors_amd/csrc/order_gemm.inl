// Products of a series with an ordinary matrix, C_o = A_o B (or A B_o), o = 0..K, as one matrix
// product in which the orders are further rows (columns) of C; and the sum of products of two series,
// C = sum_s op(A_s) op(B_s) (the gradient of an ordinary operand), in which the orders lengthen the
// contraction. float32, and bfloat16 / float16 with float32 accumulation. An ordinary operand mixes no orders, so the
// k-diagonals share nothing as they do in the series-by-series kernels (cauchy_matmul*.inl, which run the products
// that are not worth it here, order_gemm_pays): what bounds it is how fast one tile's contraction streams from memory
// to the MFMAs. With K = 3, the forward products and the input gradients of a 1024 -> 4096 -> 1024 bfloat16 layer
// pair on 4096 rows took 232 and 222 us each (600 TFLOP/s) there and take 139-144 in a training step (950-990, MFMA
// busy 46%; a forward product launched alone 123 us); 8192 rows of float32 with a bias, 768 -> 3072, 1410 us a call
// among others and 1149 (134.5 TFLOP/s, MFMA busy 85%).
//
// * Chunks of 64 bytes of contraction (32 halves, 16 floats) are moved into LDS by LDS DMA
//   (half_mfma.h) into four buffers, two chunks at a time where an operand's rows run along the
//   contraction: rows of 128 bytes, whole cache lines. A unit's DMA is issued when the operands of the
//   unit whose buffers it takes are in registers, and waited for by a count (vmcnt).
//   The rate a tile's operands arrive at is what bounds the halves: past its L2 a CU reads 64-byte
//   segments at 56-66 GB/s and 128-byte ones at 85-95 (measured with a DMA-only kernel over 16 MB), and
//   with single chunks of 64-byte rows the tiles ran at 50-57 GB/s a CU whatever the ring's depth (4, 5 or
//   8 chunks), waves (4 or 8) and order of issue. Two together: 4096 x 1024 x 4096 at degree 3 130 -> 123 us in
//   256 x 256 tiles and 177 -> 145 in 128 x 128 ones. With both operands along columns rows are longer
//   than a line as they are, and single chunks, a deeper ring, are faster (the weight gradient below,
//   before its contraction was split: 190 us, 230 in pairs).
// * Operands are read from LDS one chunk ahead into a second register set, so the LDS reads issue
//   between the MFMAs of the chunk before: one barrier per unit.
// * Operands may be stored with the contraction along rows (A [m][k], B [n][k]) or along columns
//   (A [k][m], B [k][n]), the latter read through transpose reads (halves) or element reads (floats):
//   no operand is transposed in memory. The weight gradient of the layer pair above, which ran as a
//   full series product of transposed copies (K = 3: ten pairs for the four that the one order of a
//   weight needs), took 283 us a product and 184 us of transposes, and takes 151 us (910 TFLOP/s:
//   256 tiles of 128 x 128, one a CU, the contraction in two halves).
#pragma once

#include <algorithm>
#include <type_traits>

#include "cauchy_matmul.h"
#include "half_mfma.h"
#include "mfma.h"

namespace pt {

// One MFMA block of a chunk: its operand registers per lane, and how they are read from a tile.
// Tiles with the contraction along rows: [row][64 bytes], 16-byte chunk ch of row r stored at
// ch ^ F((r / 4) % 4) with F = (0, 2, 3, 1); along columns: [k][width], chunk ^ kSwz(k).
template <typename T>
struct OrderBlock;

__host__ __device__ __forceinline__ int order_swz_rows(int r, int ch) { return ch ^ ((0x78 >> (2 * ((r >> 2) & 3))) & 3); }

template <typename T>
struct OrderBlockHalf {
  static constexpr int S = 16, ACC = 4, STEPS = 1;   // block side, accumulator registers, MFMAs per chunk
  using frag_t = u32x4;
  using acc_t = floatx4;
  // rows along n of the block are consecutive in a lane: C^T = B^T A^T
  __host__ __device__ __forceinline__ static int swz_k(int k, int ch) {   // rows of at least 256 bytes
    return ch ^ (2 * ((k & 3) | (((k >> 3) & 1) << 2)));
  }
  __device__ __forceinline__ static frag_t read_rows(const T* tile, int row0, int lane) {
    const int row = row0 + lane % 16;
    return *reinterpret_cast<const u32x4*>(&tile[row * 32 + order_swz_rows(row, lane / 16) * 8]);
  }
  template <int W>
  __device__ __forceinline__ static frag_t read_cols(const T* tile, int col0, int lane) {
    const int g = lane / 16, j = (lane % 16) / 4, a = lane % 4;
    const int k1 = 8 * g + j, k2 = 8 * g + 4 + j;
    const int ch = col0 / 8 + a / 2, e = 4 * (a % 2);
    return lds_read_tr16x2(&tile[k1 * W + swz_k(k1, ch) * 8 + e], &tile[k2 * W + swz_k(k2, ch) * 8 + e]);
  }
  __device__ __forceinline__ static acc_t zero() { return acc_t{0.f, 0.f, 0.f, 0.f}; }
  __device__ __forceinline__ static acc_t mma(const frag_t& a, const frag_t& b, int, acc_t c) {
    return HalfMfma<T>::mma(b, a, c);
  }
};
template <>
struct OrderBlock<bf16> : OrderBlockHalf<bf16> {};
template <>
struct OrderBlock<_Float16> : OrderBlockHalf<_Float16> {};

template <>
struct OrderBlock<float> {
  static constexpr int S = 32, ACC = 16, STEPS = 8;
  struct frag_t {
    float v[8];   // contraction elements 8 (lane / 32) .. + 7 of row lane % 32
  };
  using acc_t = floatx16;
  __host__ __device__ __forceinline__ static int swz_k(int k, int ch) { return ch ^ (8 * ((k >> 3) & 1)); }
  __device__ __forceinline__ static frag_t read_rows(const float* tile, int row0, int lane) {
    const int row = row0 + lane % 32, h = lane / 32;
    frag_t f;
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const Vec<float, 4> x = load_vec<float, 4>(&tile[row * 16 + order_swz_rows(row, 2 * h + q) * 4]);
#pragma unroll
      for (int e = 0; e < 4; ++e) f.v[4 * q + e] = x.v[e];
    }
    return f;
  }
  template <int W>
  __device__ __forceinline__ static frag_t read_cols(const float* tile, int col0, int lane) {
    const int col = col0 + lane % 32, h = lane / 32;
    frag_t f;
#pragma unroll
    for (int s = 0; s < 8; ++s) f.v[s] = tile[(8 * h + s) * W + swz_k(8 * h + s, col / 4) * 4 + col % 4];
    return f;
  }
  __device__ __forceinline__ static acc_t zero() { return Mfma<float>::zero(); }
  __device__ __forceinline__ static acc_t mma(const frag_t& a, const frag_t& b, int s, acc_t c) {
    return Mfma<float>::mma(b.v[s], a.v[s], c);
  }
};

template <typename T>
struct OrderGemmParams {
  CPtrs<T> a, b;
  MPtrs<T> c;
  const T* bias;                // null, or n values added to every row of order 0
  int m, n, k;                  // of one order; zeros from k to the next 16-byte vector where it runs along rows
  int lda, ldb;                 // row strides in elements
  int a_bytes, b_bytes;         // extent of one matrix
  int64_t a_bs, b_bs, c_bs;     // batch strides in elements
  int a_step, b_step;           // 1 where the operand's pointer changes by order
  int orders;                   // orders of C, or terms of a sum
  int tiles_m, tiles_n;         // of one order
};

template <typename T, int WMW, int WNW, int FM, int FN>
struct OrderTile {
  using B = OrderBlock<T>;
  static constexpr int BM = WMW * FM * B::S, BN = WNW * FN * B::S, BK = 64 / static_cast<int>(sizeof(T));
  static constexpr int kWaves = WMW * WNW, kThreads = kWaves * kWave;
  static constexpr int SA = BM / 16 / kWaves, SB = BN / 16 / kWaves;   // 1 KB DMA segments per wave and chunk
  static_assert(SA * 16 * kWaves == BM && SB * 16 * kWaves == BN, "whole DMA segments per wave");
};

template <int N>
__device__ __forceinline__ void order_wait_barrier() {   // at most N of this wave's vector loads in flight
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

template <typename T, int WMW, int WNW, int FM, int FN, bool A_COLS, bool B_COLS, bool SUM, int SPLIT, int MIN_WAVES>
__global__ __launch_bounds__(WMW* WNW* kWave* SPLIT) __attribute__((amdgpu_waves_per_eu(MIN_WAVES)))
void order_gemm_kernel(OrderGemmParams<T> p) {
  using Tile = OrderTile<T, WMW, WNW, FM, FN>;
  using Blk = OrderBlock<T>;
  constexpr int BM = Tile::BM, BN = Tile::BN, BK = Tile::BK, V = 16 / static_cast<int>(sizeof(T));
  constexpr int SA = Tile::SA, SB = Tile::SB;
  // chunks moved together, sets of them in LDS, buffers
  constexpr int UNIT = A_COLS && B_COLS ? 1 : 2, SETS = 4 / UNIT, R = UNIT * SETS;
  static_assert(static_cast<size_t>(SPLIT) * R * (BM + BN) * 64 <= 160 * 1024, "LDS budget");
  constexpr int CPA = A_COLS ? BM / V : 4, CPB = B_COLS ? BN / V : 4;   // 16-byte chunks per tile row
  __shared__ __attribute__((aligned(16))) T As[SPLIT * R][BM * BK];
  __shared__ __attribute__((aligned(16))) T Bs[SPLIT * R][BN * BK];

  const int lane = threadIdx.x % kWave;
  const int wave_id = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int wave = wave_id % Tile::kWaves;
  const int part = SPLIT == 1 ? 0 : wave_id / Tile::kWaves;   // of the contraction
  const int own = part * R;                                   // its buffers
  const int wm = wave / WNW, wn = wave % WNW;

  // Workgroup -> tile: consecutive ids go round robin over the 8 XCDs, so each XCD takes a
  // contiguous range of tiles; within it kGroup tile rows are walked column by column.
  constexpr int kXcd = 8, kGroup = 8;
  int t = blockIdx.x;
  {
    const int total = gridDim.x, per = total / kXcd;
    if (t < per * kXcd) t = (t % kXcd) * per + t / kXcd;
  }
  const int rows = p.tiles_m * (SUM || p.a_step == 0 ? 1 : p.orders);   // tile rows: every order's of A
  const int cols = p.tiles_n * (SUM || p.a_step != 0 || p.b_step == 0 ? 1 : p.orders);
  const int per_batch = rows * cols;
  const int64_t batch = t / per_batch;
  t %= per_batch;
  const int group = t / (kGroup * cols), first = group * kGroup, high = min(kGroup, rows - first);
  const int tr = first + (t % (kGroup * cols)) % high, tc = (t % (kGroup * cols)) / high;
  const int oa = tr / p.tiles_m, ob = tc / p.tiles_n;   // (one of them is 0)
  const int tile_m = (tr % p.tiles_m) * BM, tile_n = (tc % p.tiles_n) * BN;
  const int order = SUM ? 0 : oa + ob;

  // this wave's DMA segments: each lane's byte offset in the matrix and contraction position in
  // the chunk (past every chunk's end for rows and columns outside the matrix)
  int va[SA], vb[SB], ka[SA], kb[SB];
#pragma unroll
  for (int s = 0; s < SA; ++s) {
    const int slot = (wave * SA + s) * 64 + lane, r = slot / CPA, ch = slot % CPA;
    if constexpr (A_COLS) {
      const int lch = Blk::swz_k(r, ch), g = tile_m + lch * V;
      va[s] = (r * p.lda + g) * static_cast<int>(sizeof(T));
      ka[s] = g < p.m ? r : INT32_MAX;
    } else {
      const int lch = order_swz_rows(r, ch), g = tile_m + r;
      va[s] = (g * p.lda + lch * V) * static_cast<int>(sizeof(T));
      ka[s] = g < p.m ? lch * V : INT32_MAX;
    }
  }
#pragma unroll
  for (int s = 0; s < SB; ++s) {
    const int slot = (wave * SB + s) * 64 + lane, r = slot / CPB, ch = slot % CPB;
    if constexpr (B_COLS) {
      const int lch = Blk::swz_k(r, ch), g = tile_n + lch * V;
      vb[s] = (r * p.ldb + g) * static_cast<int>(sizeof(T));
      kb[s] = g < p.n ? r : INT32_MAX;
    } else {
      const int lch = order_swz_rows(r, ch), g = tile_n + r;
      vb[s] = (g * p.ldb + lch * V) * static_cast<int>(sizeof(T));
      kb[s] = g < p.n ? lch * V : INT32_MAX;
    }
  }
  const int step_a = (A_COLS ? BK * p.lda : BK) * static_cast<int>(sizeof(T));
  const int step_b = (B_COLS ? BK * p.ldb : BK) * static_cast<int>(sizeof(T));
  const int per_term = (p.k + UNIT * BK - 1) / (UNIT * BK);   // units
  const int units = ((SUM ? per_term * p.orders : per_term) + SPLIT - 1) / SPLIT;   // of a part

  // The unit to issue next: its term of the sum, its position, its buffers. Past the last one every lane
  // is out of range (zeros nobody reads), so each unit counts the same loads.
  int is = 0, ip = 0, ibuf = 0, left = p.k;
  if constexpr (SPLIT > 1) {   // (k > 0)
    is = part * units / per_term;
    ip = part * units % per_term;
    left = is < (SUM ? p.orders : 1) ? p.k - ip * UNIT * BK : 0;
#pragma unroll
    for (int s = 0; s < SA; ++s) va[s] += ip * UNIT * step_a;
#pragma unroll
    for (int s = 0; s < SB; ++s) vb[s] += ip * UNIT * step_b;
  }
  BufferRsrc ra, rb;
  auto point = [&]() {   // the operands of term is (of order oa, ob)
    const int term = min(is, p.orders - 1);
    const int sa = SUM ? term : oa, sb = SUM ? term : ob;
    ra = buffer_rsrc(p.a.p[sa] + batch * p.a_bs, p.a_bytes);
    rb = buffer_rsrc(p.b.p[sb] + batch * p.b_bs, p.b_bytes);
  };
  point();
  auto issue_segment = [&](int i) {   // i / UNIT: the segment, A's SA then B's SB; i % UNIT: the chunk
    const int s = i / UNIT, half = i % UNIT;
    if (s < SA) {
      lds_dma16(&As[own + ibuf + half][(wave * SA + s) * (1024 / static_cast<int>(sizeof(T)))], ra,
                ka[s] < left - half * BK ? va[s] : kBufferOutOfRange);
      va[s] += step_a;
    } else {
      const int u = s - SA;
      lds_dma16(&Bs[own + ibuf + half][(wave * SB + u) * (1024 / static_cast<int>(sizeof(T)))], rb,
                kb[u] < left - half * BK ? vb[u] : kBufferOutOfRange);
      vb[u] += step_b;
    }
  };
  auto issued = [&]() {
    ibuf = ibuf + UNIT == R ? 0 : ibuf + UNIT;
    left -= UNIT * BK;
    if (++ip == per_term) {
      ip = 0;
      ++is;
      left = SUM && is < p.orders ? p.k : 0;
      if constexpr (SUM) {
#pragma unroll
        for (int s = 0; s < SA; ++s) va[s] -= UNIT * per_term * step_a;
#pragma unroll
        for (int s = 0; s < SB; ++s) vb[s] -= UNIT * per_term * step_b;
        point();
      }
    }
  };

  typename Blk::acc_t acc[FM][FN];
#pragma unroll
  for (int fm = 0; fm < FM; ++fm)
#pragma unroll
    for (int fn = 0; fn < FN; ++fn) acc[fm][fn] = Blk::zero();

  typename Blk::frag_t fa[2][FM], fb[2][FN];
  auto read_operand = [&](int buf, int set, int i) {   // operand i of a chunk: B's FN, then A's FM
    if (i < FN) {
      const int at = (wn * FN + i) * Blk::S;
      if constexpr (B_COLS) fb[set][i] = Blk::template read_cols<BN>(Bs[own + buf], at, lane);
      else fb[set][i] = Blk::read_rows(Bs[own + buf], at, lane);
    } else {
      const int at = (wm * FM + i - FN) * Blk::S;
      if constexpr (A_COLS) fa[set][i - FN] = Blk::template read_cols<BM>(As[own + buf], at, lane);
      else fa[set][i - FN] = Blk::read_rows(As[own + buf], at, lane);
    }
  };
  auto multiply_row = [&](int set, int fm) {
#pragma unroll
    for (int s = 0; s < Blk::STEPS; ++s)   // (no MFMA waits for the one before it)
#pragma unroll
      for (int fn = 0; fn < FN; ++fn) acc[fm][fn] = Blk::mma(fa[set][fm], fb[set][fn], s, acc[fm][fn]);
  };

  constexpr int LOADS = UNIT * (SA + SB);   // of a unit
  for (int i = 0; i < SETS; ++i) {
#pragma unroll
    for (int s = 0; s < LOADS; ++s) issue_segment(s);
    issued();
  }
  order_wait_barrier<(SETS - 1) * LOADS>();   // unit 0 has landed, for every wave
#pragma unroll
  for (int i = 0; i < FM + FN; ++i) read_operand(0, 0, i);
  // One chunk: its MFMAs from register set `set`, the operand reads of the next chunk from `buf`, and in
  // the last chunk of unit j the DMA of unit j + SETS into the buffers of this one. The reads and the
  // DMA are spread between the MFMA rows (fixed by the scheduling barriers).
  auto step = [&](int set, int buf, bool issue) {
#pragma unroll
    for (int fm = 0; fm < FM; ++fm) {
      multiply_row(set, fm);
#pragma unroll
      for (int i = fm * (FM + FN) / FM; i < (fm + 1) * (FM + FN) / FM; ++i) read_operand(buf, set ^ 1, i);
      if (issue) {
#pragma unroll
        for (int s = fm * LOADS / FM; s < (fm + 1) * LOADS / FM; ++s) issue_segment(s);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  int buf = 0;
  auto last_of_unit = [&](int set) {
    order_wait_barrier<(SETS - 2) * LOADS>();   // unit j + 1 has landed; every wave has read unit j
    buf = buf + UNIT == R ? 0 : buf + UNIT;
    step(set, buf, true);
    issued();
  };
  if constexpr (UNIT == 2) {
    for (int j = 0; j < units; ++j) {
      step(0, buf + 1, false);
      last_of_unit(1);
    }
  } else {
    int j = 0;
    for (; j + 1 < units; j += 2) {
      last_of_unit(0);
      last_of_unit(1);
    }
    if (j < units) last_of_unit(0);
  }
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");   // no DMA outlives the workgroup's LDS

  if constexpr (SPLIT == 2) {   // the second part's sums go to the first through LDS (every wave is done with its tiles)
    static_assert(Blk::ACC == 4 && FM * FN * Tile::kThreads * 16 <= sizeof(As), "sums fit A's buffers");
    const int at = threadIdx.x % Tile::kThreads;
    __syncthreads();
    if (part == 1) {
#pragma unroll
      for (int i = 0; i < FM * FN; ++i)
        reinterpret_cast<floatx4*>(&As[0][0])[i * Tile::kThreads + at] = acc[i / FN][i % FN];
    }
    __syncthreads();
    if (part == 1) return;
#pragma unroll
    for (int i = 0; i < FM * FN; ++i)
      acc[i / FN][i % FN] += reinterpret_cast<const floatx4*>(&As[0][0])[i * Tile::kThreads + at];
  }

  // ---- epilogue: a lane's registers are runs of four columns of one row of C ----
  T* base = p.c.p[order] + batch * p.c_bs;
  const int row0 = tile_m + wm * FM * Blk::S + lane % Blk::S;
  const int col0 = tile_n + wn * FN * Blk::S + 4 * (lane / Blk::S);   // of block 0 and its registers 0..3
  auto store = [&](auto biased) __attribute__((always_inline)) {
    float add[FN][Blk::ACC];
    if constexpr (decltype(biased)::value) {   // before the stores: between them the loads would wait for the ones issued
#pragma unroll
      for (int fn = 0; fn < FN; ++fn)
#pragma unroll
        for (int i = 0; i < Blk::ACC; ++i) {
          const int col = col0 + fn * Blk::S + 8 * (i / 4) + i % 4;
          add[fn][i] = col < p.n ? to_acc(p.bias[col]) : 0.f;
        }
    }
#pragma unroll
    for (int fm = 0; fm < FM; ++fm) {
      const int row = row0 + fm * Blk::S;
      if (row >= p.m) continue;
#pragma unroll
      for (int fn = 0; fn < FN; ++fn)
#pragma unroll
        for (int q = 0; q < Blk::ACC / 4; ++q) {
          const int col = col0 + fn * Blk::S + 8 * q;
          float v[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            v[e] = acc[fm][fn][4 * q + e];
            if constexpr (decltype(biased)::value) v[e] += add[fn][4 * q + e];
          }
          T* dst = base + static_cast<int64_t>(row) * p.n + col;
          if (col + 3 < p.n) {
            Vec<T, 4> w;
#pragma unroll
            for (int e = 0; e < 4; e += 2) vec_put2(w, e, v[e], v[e + 1]);
            __builtin_memcpy(dst, &w, sizeof(w));   // at any element: one 8- or 16-byte store
            // (else the compiler shares the element stores below and splits this one: 4 x 3000 x 16 x 2048
            // float32 at degree 1 takes 92 us with stores of 12 and 4 bytes, 66 with whole ones)
            asm volatile("" ::: "memory");
          } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
              if (col + e < p.n) dst[e] = from_acc<T>(v[e]);
          }
        }
    }
  };
  if (p.bias != nullptr && order == 0) store(std::true_type{});
  else store(std::false_type{});
}

// Whether a launch holds this many tiles for each order and batch entry: every workgroup has 256 threads
// at least counted so (the larger tiles and the split ones, of 512, are fewer), and a launch has fewer
// than 2^32 threads along x.
template <typename T>
static bool order_gemm_holds(int64_t m, int64_t n, int64_t count) {
  constexpr int64_t side = sizeof(T) == 2 ? 128 : 64;   // of the smallest tile
  return static_cast<double>((m + side - 1) / side) * static_cast<double>((n + side - 1) / side) * static_cast<double>(count) <
         static_cast<double>(1 << 24);
}

// Whether the kernel can run the product: whole, aligned 16-byte vectors along rows, 32-bit offsets, one launch.
template <typename T>
static bool order_gemm_takes(const CauchyArgs& a) {
  constexpr int64_t V = 16 / static_cast<int64_t>(sizeof(T)), kLimit = (int64_t{1} << 30) / static_cast<int64_t>(sizeof(T));
  bool ok = a.lda % V == 0 && a.ldb % V == 0 && a.a_bs % V == 0 && a.b_bs % V == 0 && a.lda < kLimit && a.ldb < kLimit &&
            a.m * a.lda < kLimit && a.rows_b() * a.ldb < kLimit &&
            order_gemm_holds<T>(a.m, a.n, std::max(a.a_orders, a.b_orders) * a.batch);
  for (int o = 0; o < a.a_orders; ++o) ok = ok && pt_host::aligned16(a.a[o]);
  for (int o = 0; o < a.b_orders; ++o) ok = ok && pt_host::aligned16(a.b[o]);
  return ok;
}

template <typename T, int WMW, int WNW, int FM, int FN, bool A_COLS, bool B_COLS, bool SUM, int SPLIT = 1>
static int launch_order_tile(OrderGemmParams<T> p, int64_t batch, hipStream_t stream) {
  using Tile = OrderTile<T, WMW, WNW, FM, FN>;
  p.tiles_m = (p.m + Tile::BM - 1) / Tile::BM;
  p.tiles_n = (p.n + Tile::BN - 1) / Tile::BN;
  const int64_t tiles = static_cast<int64_t>(p.tiles_m) * p.tiles_n * (SUM ? 1 : p.orders) * batch;
  order_gemm_kernel<T, WMW, WNW, FM, FN, A_COLS, B_COLS, SUM, SPLIT, 2>
      <<<dim3(static_cast<unsigned>(tiles)), dim3(SPLIT * Tile::kThreads), 0, stream>>>(p);
  PT_LAUNCH_CHECK();
  return PT_OK;
}

// The tile: the one with the least estimated time per chunk of contraction over the launch.
// * Halves: 256 x 256 (one workgroup of 8 waves a CU) takes 0.80 us a chunk with every CU busy, and
//   128 x 128 (up to two workgroups of 4 waves a CU) 0.49 us with two and 0.34 with one (from 8192^3
//   at 820 and 1007 us, and 512 chunks of 256 small tiles at 176 us): four small tiles cost 1.2
//   times a large one where both fill the chip, less where the large ones leave CUs idle. Up to 256
//   small tiles, one a CU, run as workgroups of 8 waves, each half of which takes half of the contraction:
//   the chunks of both then arrive at the rate of two tiles a CU. From 8 chunks a half, below which the
//   sums' way through LDS is not paid for (weight gradients of 4096 rows, 1024 x 4096, degree 3: 190 -> 151 us).
// * Floats: 128 x 128, 128 x 64 and 64 x 64 (two, three and five workgroups a CU); MFMA-bound, so the
//   busiest CU's tiles count, at 137, 133 and 128 TFLOP/s (8192 x 768 x 3072, degree 3).
static inline bool order_large_tiles(int64_t large, int64_t small) {
  const int64_t rest = small % 512;
  return 0.80 * static_cast<double>((large + 255) / 256) <
         0.49 * static_cast<double>(small / 512) + (rest == 0 ? 0.0 : rest <= 256 ? 0.34 : 0.49);
}

static inline int order_float_tile(const int64_t (&tiles)[3]) {   // 0: 128 x 128, 1: 128 x 64, 2: 64 x 64
  constexpr double kArea[3] = {128 * 128, 128 * 64, 64 * 64}, kRate[3] = {137, 133, 128};
  double cost[3];
  for (int i = 0; i < 3; ++i) cost[i] = static_cast<double>((tiles[i] + 255) / 256) * kArea[i] / kRate[i];
  return cost[0] <= cost[1] && cost[0] <= cost[2] ? 0 : cost[1] <= cost[2] ? 1 : 2;
}

template <typename T, bool A_COLS, bool B_COLS, bool SUM>
static int launch_order_gemm(const OrderGemmParams<T>& p, int64_t batch, hipStream_t stream) {
  auto tiles = [&](int64_t bm, int64_t bn) {
    return (p.m + bm - 1) / bm * ((p.n + bn - 1) / bn) * (SUM ? 1 : p.orders) * batch;
  };
  if constexpr (sizeof(T) == 2) {
    const int64_t small = tiles(128, 128), chunks = (p.k + 31) / 32 * (SUM ? p.orders : 1);
    if (small <= 256 && chunks >= 16) return launch_order_tile<T, 2, 2, 4, 4, A_COLS, B_COLS, SUM, 2>(p, batch, stream);
    if (order_large_tiles(tiles(256, 256), small)) return launch_order_tile<T, 2, 4, 8, 4, A_COLS, B_COLS, SUM>(p, batch, stream);
    return launch_order_tile<T, 2, 2, 4, 4, A_COLS, B_COLS, SUM>(p, batch, stream);
  } else {
    const int64_t t[3] = {tiles(128, 128), tiles(128, 64), tiles(64, 64)};
    switch (order_float_tile(t)) {
      case 0: return launch_order_tile<T, 2, 2, 2, 2, A_COLS, B_COLS, SUM>(p, batch, stream);
      case 1: return launch_order_tile<T, 2, 2, 2, 1, A_COLS, B_COLS, SUM>(p, batch, stream);
      default: return launch_order_tile<T, 2, 2, 1, 1, A_COLS, B_COLS, SUM>(p, batch, stream);
    }
  }
}

// Whether the product runs order by order rather than in the kernels with all orders in a workgroup
// (cauchy_matmul*.inl): those read an ordinary tile once for all orders and have smaller tiles, this one streams a
// long contraction faster. The estimated times of both in us: a fixed part, and for every round of workgroups
// over the chip one for the stores and one for every 32 (floats: 16) of the contraction; fitted to 2400 products
// (sides 1 to 100000, contractions 8 to 4096, 1 to 16384 matrices, degrees 1 to 8; 1e4 to 1e12 multiply-adds),
// whose times they give to 7-9% (floats) and 13-20%. Order by order where it is less (halves: by 10%): then 2% of
// the products take over 1.08 times what the other kernel takes; always order by order 45% do, up to 8 times (4096
// x 16 x 16 x 16 bfloat16, degree 8: 40 us and 202; 200000 x 8 x 8, 53 and 129; 2048 x 8 x 2048 float32, degree 3, 17
// and 30; the other way 768 x 4096 x 256 bfloat16, degree 8, 104 and 40; 8192 x 768 x 3072 float32, 1350 and 1150).
template <typename T>
static bool order_gemm_pays(const CauchyArgs& a) {
  const int64_t orders = std::max(a.a_orders, a.b_orders);
  const double n1 = static_cast<double>(orders);
  auto tiles = [&](int64_t bm, int64_t bn) { return (a.m + bm - 1) / bm * ((a.n + bn - 1) / bn) * a.batch; };
  auto whole_rounds = [](int64_t count) { return static_cast<double>((count + 255) / 256); };
  // rounds of 512 workgroups; `half` of one where the last has at most half of them
  auto rounds = [](int64_t count, double half) {
    const int64_t rest = count % 512;
    return static_cast<double>(count / 512) + (rest == 0 ? 0.0 : rest <= 256 ? half : 1.0);
  };
  if constexpr (sizeof(T) == 2) {
    const double chunks = static_cast<double>((a.k + 31) / 32);
    const double all = orders <= 5 && a.m >= 256 && a.n >= 256
        ? 2.4 + whole_rounds(tiles(128, 128)) * (2.0 * n1 + chunks * (0.075 + 0.23 * n1))
        : 2.4 + rounds(tiles(64, 64), 0.44) * (0.94 * n1 + chunks * (0.17 + 0.17 * n1));
    const int64_t small = tiles(128, 128) * orders, large = tiles(256, 256) * orders;
    double each;   // (the tiles as launch_order_gemm picks them)
    if (small <= 256 && chunks >= 16) each = 6.2 + 0.20 * chunks;
    else if (order_large_tiles(large, small)) each = 3.7 + whole_rounds(large) * (9.8 + 0.77 * chunks);
    else each = 3.7 + rounds(small, 0.46) * (3.9 + 0.47 * chunks);
    return 1.10 * each <= all;
  } else {
    const double chunks = static_cast<double>((a.k + 15) / 16);
    const double all = 2.3 + rounds(tiles(64, 64), 0.56) * (0.97 * n1 + chunks * (0.125 + 0.53 * n1));
    const int64_t t[3] = {tiles(128, 128) * orders, tiles(128, 64) * orders, tiles(64, 64) * orders};
    const int pick = order_float_tile(t);
    constexpr double kStores[3] = {3.6, 1.54, 0.76}, kOne[3] = {1.05, 0.59, 0.30}, kMany[3] = {0.96, 0.51, 0.27};
    const double q = whole_rounds(t[pick]);   // tiles of the busiest CU
    return 3.2 + q * kStores[pick] + chunks * (q == 1.0 ? kOne[pick] : q * kMany[pick]) <= all;
  }
}

// C_o = A_o B or A B_o for `orders` orders (operands with one order are shared by all).
template <typename T>
static int launch_by_order(const CauchyArgs& a, int orders) {
  OrderGemmParams<T> p{};
  for (int o = 0; o < a.a_orders; ++o) p.a.p[o] = static_cast<const T*>(a.a[o]);
  for (int o = 0; o < a.b_orders; ++o) p.b.p[o] = static_cast<const T*>(a.b[o]);
  for (int o = 0; o < orders; ++o) p.c.p[o] = static_cast<T*>(a.c[o]);
  p.bias = static_cast<const T*>(a.bias);
  p.m = static_cast<int>(a.m);
  p.n = static_cast<int>(a.n);
  p.k = static_cast<int>(a.k);
  p.lda = static_cast<int>(a.lda);
  p.ldb = static_cast<int>(a.ldb);
  p.a_bytes = static_cast<int>(a.m * a.lda * static_cast<int64_t>(sizeof(T)));
  p.b_bytes = static_cast<int>(a.rows_b() * a.ldb * static_cast<int64_t>(sizeof(T)));
  p.a_bs = a.a_bs;
  p.b_bs = a.b_bs;
  p.c_bs = a.m * a.n;
  p.a_step = a.a_orders > 1;
  p.b_step = a.b_orders > 1;
  p.orders = orders;
  if (a.trans_b) return launch_order_gemm<T, false, false, false>(p, a.batch, a.stream);
  return launch_order_gemm<T, false, true, false>(p, a.batch, a.stream);
}

template <typename T>
int launch_order_sum(const OrderSumArgs& a) {
  constexpr int64_t V = 16 / static_cast<int64_t>(sizeof(T)), kLimit = (int64_t{1} << 30) / static_cast<int64_t>(sizeof(T));
  const int64_t rows_a = a.trans_a ? a.k : a.m, rows_b = a.trans_b ? a.n : a.k;
  bool ok = a.lda % V == 0 && a.ldb % V == 0 && a.a_bs % V == 0 && a.b_bs % V == 0 &&
            a.m <= INT32_MAX && a.n <= INT32_MAX && a.k <= INT32_MAX &&
            a.lda < kLimit && a.ldb < kLimit && rows_a * a.lda < kLimit && rows_b * a.ldb < kLimit &&
            order_gemm_holds<T>(a.m, a.n, a.batch);
  for (int s = 0; s < a.terms; ++s) ok = ok && pt_host::aligned16(a.a[s]) && pt_host::aligned16(a.b[s]);
  if (!ok) {
    pt_host::set_error("matmul order sum: needs 16-byte aligned operands, row and batch strides of whole 16-byte "
                       "vectors, and each matrix below 1 GiB, and tiles of one launch");
    return PT_UNSUPPORTED;
  }
  OrderGemmParams<T> p{};
  for (int s = 0; s < a.terms; ++s) {
    p.a.p[s] = static_cast<const T*>(a.a[s]);
    p.b.p[s] = static_cast<const T*>(a.b[s]);
  }
  p.c.p[0] = static_cast<T*>(a.c);
  p.m = static_cast<int>(a.m);
  p.n = static_cast<int>(a.n);
  p.k = static_cast<int>(a.k);
  p.lda = static_cast<int>(a.lda);
  p.ldb = static_cast<int>(a.ldb);
  p.a_bytes = static_cast<int>(rows_a * a.lda * static_cast<int64_t>(sizeof(T)));
  p.b_bytes = static_cast<int>(rows_b * a.ldb * static_cast<int64_t>(sizeof(T)));
  p.a_bs = a.a_bs;
  p.b_bs = a.b_bs;
  p.c_bs = a.m * a.n;
  p.a_step = p.b_step = 1;
  p.orders = a.terms;
  if (a.trans_a) return launch_order_gemm<T, true, true, true>(p, a.batch, a.stream);
  if (a.trans_b) return launch_order_gemm<T, false, false, true>(p, a.batch, a.stream);
  return launch_order_gemm<T, false, true, true>(p, a.batch, a.stream);
}

}  // namespace pt
