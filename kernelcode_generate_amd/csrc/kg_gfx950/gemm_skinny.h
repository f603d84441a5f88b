// gemm_skinny_kernel: matmul of few rows (bf16, f16, fp32), bound by the reading of rhs. Any
// M >= 1, N >= 2 and K >= 1, any row strides and bases of whole elements.
//
// A workgroup of 16 waves takes 32 columns and 16 or 32 rows, each wave every 16th piece of 64 k: its
// lanes load rhs straight into registers, two columns by eight k-rows each (a wave's load is
// four row segments of 32 columns), with the next 64 k in flight under the MFMAs of the last;
// K needs neither an LDS ring nor barriers. The k-rows of one column are put together by
// v_perm_b32 (16-bit), and the two columns of a lane go to two v_mfma_f32_16x16x32 (fp32: to
// 2 x 8 of 16x16x4). One LDS sum over the 16 waves, by halves, ends the call: no fp32 partials
// in HBM and no second launch. Neighbouring workgroups,
// which share the 128-byte lines of rhs rows (and, of more rows, all of rhs), run on one XCD,
// whose L2 fetches each line once. Pieces of 64 k, not 32, read whole lines of 16-bit lhs rows.
//
// Measured (us, before / this kernel; the call itself costs 6.8): bf16 16x4096x4096 14.9 / 11.7
// (2.9 TB/s; one row: 12.4 / 8.1, 4.1 TB/s), 16x8192x8192 28.3 / 26.0 (5.2 TB/s), 64x512x4096
// 13.2 / 7.4, odd 16x8001x8001 129 / 37; fp32 16x4096x4096 302 / 18, 64x8192x8192 604 / 120. Half of the CUs
// have no tile at N = 4096: two workgroups on one tile's K would need partials in HBM.
#pragma once

#include "common.h"
#include "conv2d_igemm.h"  // F32Tag, IgElem

namespace kg_gfx950 {

namespace gemms {
constexpr int kCols = 32;      // columns per workgroup
constexpr int kWaves = 16;
constexpr int kStep = 32;      // k per step
constexpr int kDepth = 2;      // steps per batch: 128-byte lines of 16-bit lhs rows

typedef uint32_t u32_any __attribute__((aligned(2)));
typedef u32x2 u32x2_any __attribute__((aligned(4)));
typedef u32x4 u32x4_any16 __attribute__((aligned(2)));
typedef u32x4 u32x4_any32 __attribute__((aligned(4)));

template <typename Tag>
struct Step {  // 16-bit: a lane's 8 k of each of its rows, two columns of each of its 8 k-rows
  template <int kMT>
  struct Regs {
    u32x4 a[kMT];
    uint32_t b[8];
  };
  static __device__ __forceinline__ uint32_t load_b(const char* p) { return *reinterpret_cast<const u32_any*>(p); }
  template <int kMT>
  static __device__ __forceinline__ void load_a(Regs<kMT>& r, int i, const char* p) {
    r.a[i] = *reinterpret_cast<const u32x4_any16*>(p);
  }
  template <int kMT>
  static __device__ __forceinline__ void set_a(Regs<kMT>& r, int i, const uint16_t v[8]) {
#pragma unroll
    for (int q = 0; q < 4; ++q) r.a[i][q] = pack16(v[2 * q], v[2 * q + 1]);
  }
  template <int kMT>
  static __device__ __forceinline__ void mac(const Regs<kMT>& r, f32x4 (&acc)[kMT][2]) {
    u32x4 c0, c1;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      c0[q] = lo_halves(r.b[2 * q], r.b[2 * q + 1]);
      c1[q] = hi_halves(r.b[2 * q], r.b[2 * q + 1]);
    }
#pragma unroll
    for (int i = 0; i < kMT; ++i) {
      acc[i][0] = Half16<Tag>::mfma16(r.a[i], c0, acc[i][0]);
      acc[i][1] = Half16<Tag>::mfma16(r.a[i], c1, acc[i][1]);
    }
  }
};

template <>
struct Step<F32Tag> {
  template <int kMT>
  struct Regs {
    u32x4 a[kMT][2];
    u32x2 b[8];
  };
  static __device__ __forceinline__ u32x2 load_b(const char* p) { return *reinterpret_cast<const u32x2_any*>(p); }
  template <int kMT>
  static __device__ __forceinline__ void load_a(Regs<kMT>& r, int i, const char* p) {
    r.a[i][0] = *reinterpret_cast<const u32x4_any32*>(p);
    r.a[i][1] = *reinterpret_cast<const u32x4_any32*>(p + 16);
  }
  template <int kMT>
  static __device__ __forceinline__ void set_a(Regs<kMT>& r, int i, const float v[8]) {
#pragma unroll
    for (int e = 0; e < 8; ++e) r.a[i][e >> 2][e & 3] = __builtin_bit_cast(uint32_t, v[e]);
  }
  // MFMA e of a step takes k = 8 (lane/16) + e of both operands
  template <int kFirst, int kMT>
  static __device__ __forceinline__ void mac_half(const Regs<kMT>& r, f32x4 (&part)[kMT][2]) {
#pragma unroll
    for (int i = 0; i < kMT; ++i) part[i][0] = part[i][1] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int e = kFirst; e < kFirst + 4; ++e)
#pragma unroll
      for (int i = 0; i < kMT; ++i) {
        const float a = __builtin_bit_cast(float, (uint32_t)r.a[i][e >> 2][e & 3]);
#pragma unroll
        for (int j = 0; j < 2; ++j)
          part[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, __builtin_bit_cast(float, (uint32_t)r.b[e][j]), part[i][j], 0, 0, 0);
      }
  }
  // chains of four MFMAs, each then added to the total: short chains round less
  template <int kMT>
  static __device__ __forceinline__ void mac(const Regs<kMT>& r, f32x4 (&acc)[kMT][2]) {
    f32x4 part[kMT][2];
    mac_half<0>(r, part);
#pragma unroll
    for (int i = 0; i < kMT; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) acc[i][j] += part[i][j];
    mac_half<4>(r, part);
#pragma unroll
    for (int i = 0; i < kMT; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) acc[i][j] += part[i][j];
  }
};
}  // namespace gemms

template <typename Tag, int kMT>  // kMT: 16-row blocks of a workgroup
__global__ __launch_bounds__(gemms::kWaves * 64) void gemm_skinny_kernel(
    const typename convg::IgElem<Tag>::T* __restrict__ A, const typename convg::IgElem<Tag>::T* __restrict__ B,
    typename convg::IgElem<Tag>::T* __restrict__ C, const void* __restrict__ bias, int bias_kind, int M, int N, int K,
    long long lda, long long ldb, long long ldc) {
  using namespace gemms;
  using E = convg::IgElem<Tag>;
  using T = typename E::T;
  using S = Step<Tag>;
  using Regs = typename S::template Regs<kMT>;
  constexpr int kRows = 16 * kMT;
  __shared__ __attribute__((aligned(16))) f32x2 red[kWaves][kRows][kCols / 2];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l16 = lane & 15, lg = lane >> 4;
  const int total = gridDim.x, xcd = blockIdx.x % 8;
  const int logical = xcd * (total / 8) + min(xcd, total % 8) + blockIdx.x / 8;
  const int row_blocks = (M + kRows - 1) / kRows;
  const int m0 = logical % row_blocks * kRows, rows = M - m0;  // rows: of this block on
  const int n0 = logical / row_blocks * kCols;
  A += m0 * lda;
  C += m0 * ldc;
  // lanes past the last column pair repeat it (their outputs are dropped), rows past M row M - 1
  const uint32_t b_off = (uint32_t)((lg * 8 * ldb + min(n0 + 2 * l16, N - 2)) * sizeof(T));
  uint32_t a_off[kMT];
#pragma unroll
  for (int i = 0; i < kMT; ++i) a_off[i] = (uint32_t)((min(16 * i + l16, rows - 1) * lda + lg * 8) * sizeof(T));

  f32x4 acc[kMT][2];
#pragma unroll
  for (int i = 0; i < kMT; ++i) acc[i][0] = acc[i][1] = f32x4{0.f, 0.f, 0.f, 0.f};

  auto load = [&](int step, Regs& r) __attribute__((always_inline)) {
    const long long k = (long long)step * kStep;
    const char* b = reinterpret_cast<const char*>(B + k * ldb);
    const char* a = reinterpret_cast<const char*>(A + k);
#pragma unroll
    for (int e = 0; e < 8; ++e) r.b[e] = S::load_b(b + e * ldb * (long long)sizeof(T) + b_off);
#pragma unroll
    for (int i = 0; i < kMT; ++i) S::load_a(r, i, a + a_off[i]);
  };

  // whole batches of 64 k: wave, wave + 16, ...; two batches' registers in turn
  const int full = K / (kDepth * kStep);
  const int batches = full > wave ? (full - wave + kWaves - 1) / kWaves : 0;
  Regs r[2][kDepth];
  auto load_batch = [&](int t, Regs (&batch)[kDepth]) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < kDepth; ++u) load((wave + kWaves * t) * kDepth + u, batch[u]);
  };
  auto mac_batch = [&](const Regs (&batch)[kDepth]) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < kDepth; ++u) S::mac(batch[u], acc);
  };
  if (batches > 0) load_batch(0, r[0]);
  int t = 0;
  for (; t + 2 < batches; t += 2) {
    load_batch(t + 1, r[1]);
    mac_batch(r[0]);
    load_batch(t + 2, r[0]);
    mac_batch(r[1]);
  }
  if (t + 1 < batches) {
    load_batch(t + 1, r[1]);
    mac_batch(r[0]);
    mac_batch(r[1]);
  } else if (t < batches) {
    mac_batch(r[0]);
  }
  // the last K % 64: zeros for k >= K in both operands (no load past the last row)
  if (wave == full % kWaves)
    for (int ks = full * kDepth * kStep; ks < K; ks += kStep) {
      const int k0 = ks + 8 * lg;
      Regs& p = r[0][0];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        auto v = S::load_b(reinterpret_cast<const char*>(B + min(k0 + e, K - 1) * ldb + min(n0 + 2 * l16, N - 2)));
        if (k0 + e >= K) v = decltype(v){};
        p.b[e] = v;
      }
#pragma unroll
      for (int i = 0; i < kMT; ++i) {
        const T* row = A + min(16 * i + l16, rows - 1) * lda;
        T v[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = k0 + e < K ? row[min(k0 + e, K - 1)] : T(0);
        S::set_a(p, i, v);
      }
      S::mac(p, acc);
    }

  // lane holds C[m = 16 i + 4 lg + e][columns 2 l16, 2 l16 + 1]
#pragma unroll
  for (int i = 0; i < kMT; ++i)
#pragma unroll
    for (int e = 0; e < 4; ++e) red[wave][16 * i + 4 * lg + e][l16] = f32x2{acc[i][0][e], acc[i][1][e]};
  __syncthreads();
  if (threadIdx.x >= kRows * (kCols / 2)) return;
  const int m = threadIdx.x / (kCols / 2), c = threadIdx.x % (kCols / 2);
  const int n = n0 + 2 * c, nb = min(n, N - 2);
  if (m >= rows || n >= N) return;
  f32x2 sum[kWaves];
#pragma unroll
  for (int w = 0; w < kWaves; ++w) sum[w] = red[w][m][c];
#pragma unroll
  for (int half = kWaves / 2; half > 0; half /= 2)
#pragma unroll
    for (int w = 0; w < half; ++w) sum[w] += sum[w + half];
  float v0 = sum[0][0], v1 = sum[0][1];
  if (bias_kind == 1) {
    v0 += static_cast<const float*>(bias)[nb];
    v1 += static_cast<const float*>(bias)[nb + 1];
  } else if (bias_kind == 2) {
    v0 += E::to_float(static_cast<const T*>(bias)[nb]);
    v1 += E::to_float(static_cast<const T*>(bias)[nb + 1]);
  }
  T* out = C + m * ldc + nb;
  T o0, o1;
  if constexpr (E::kPerChunk == 8) {
    const uint32_t packed = Half16<Tag>::pack2(v0, v1);
    o0 = (T)(packed & 0xffffu);
    o1 = (T)(packed >> 16);
  } else {
    o0 = v0;
    o1 = v1;
  }
  if (n == nb) out[0] = o0;  // otherwise N is odd and the pair to the left stores that column
  out[1] = o1;
}

// Rows per workgroup: 16 while such blocks make one round on the 256 CUs, 32 above, where reading
// rhs again for each block costs more (us, 16 / 32: bf16 64x512x4096 7.4 / 10.9, 48x1920x4096
// 8.1 / 11.3; 64x4096x4096 18.6 / 14.9, 64x8192x8192 65 / 50).
inline int gemm_skinny_rows(long long M, long long N) {
  return M <= 16 || (N + gemms::kCols - 1) / gemms::kCols * ((M + 15) / 16) <= 256 ? 16 : 32;
}

// bias_kind: 0 none, 1 fp32, 2 16-bit.
template <typename Tag>
hipError_t launch_gemm_skinny(const void* A, const void* B, void* C, const void* bias, int bias_kind, int M, int N, int K,
                              long long lda, long long ldb, long long ldc, hipStream_t stream) {
  using T = typename convg::IgElem<Tag>::T;
  const long long tiles = ((long long)N + gemms::kCols - 1) / gemms::kCols;
#define KG_GEMM_SKINNY(MT)                                                                                             \
  hipLaunchKernelGGL((gemm_skinny_kernel<Tag, MT>), dim3((unsigned)(tiles * ((M + 16 * MT - 1) / (16 * MT)))),         \
                     dim3(gemms::kWaves * 64), 0, stream,                                                              \
                     static_cast<const T*>(A), static_cast<const T*>(B), static_cast<T*>(C), bias, bias_kind, M, N, K, \
                     lda, ldb, ldc)
  if (gemm_skinny_rows(M, N) == 16) KG_GEMM_SKINNY(1);
  else KG_GEMM_SKINNY(2);
#undef KG_GEMM_SKINNY
  return hipGetLastError();
}

}  // namespace kg_gfx950
