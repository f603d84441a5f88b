// Matmuls whose rows are not 16-byte aligned (odd N or K, odd row strides or bases), 16-bit and
// fp32, on matrix cores. out = lhs @ rhs is the 1x1 convolution of an image of K channels and N
// pixels (rhs, [K][N]) with M filters of K channels (lhs, [M][K]), so the channel-last GEMM
// computes it: one launch writes rhs as [n][k] and lhs as [m][k] into the stream's workspace,
// rows padded with zeros to 128 bytes, and conv2d_nhwc_kernel multiplies them. Larger operands
// go in pieces of rows of lhs and columns of rhs that fit the workspace.
#pragma once

#include "conv2d_nhwc.h"

namespace kg_gfx950 {

namespace gemmx {
struct Params {
  int m, n, k;         // of this piece
  long long lda, ldb;  // element strides of the rows
  long long b_last;    // last element of rhs (from its piece's base) that 16 bytes may start at
  uint32_t pitch;      // bytes per packed row
  FastDiv div_chunks;  // 16-byte chunks per packed row
  FastDiv div_cols;    // pieces of V columns of rhs
};
}  // namespace gemmx

// Blocks below b_blocks: a thread packs a block of V rows (k) x V columns of rhs, read as V row
// pieces of 16 bytes at any alignment and transposed in registers; the chunks of a column in
// neighbouring threads. A piece that crosses the row's end reads on (the columns past N are
// not used), only one that would cross the operand's end is read by elements. Other blocks:
// one chunk of a row of lhs per thread.
template <typename Tag>
__global__ __launch_bounds__(convn::kThreads) void gemm_pack_kernel(
    const typename convg::IgElem<Tag>::T* __restrict__ A, const typename convg::IgElem<Tag>::T* __restrict__ B,
    u32x4* __restrict__ ap, u32x4* __restrict__ bp, gemmx::Params s, int b_blocks) {
  using T = typename convg::IgElem<Tag>::T;
  constexpr int V = convg::IgElem<Tag>::kPerChunk;
  const int chunks = (int)s.div_chunks.d;
  if ((int)blockIdx.x < b_blocks) {
    const uint32_t idx = blockIdx.x * convn::kThreads + threadIdx.x;
    const uint32_t piece = fdiv(idx, s.div_chunks);
    const int kc = (int)(idx - piece * chunks), k0 = kc * V;
    const int n0 = (int)piece * V;
    if (n0 >= s.n) return;
    u32x4 in[V], out[V];
#pragma unroll
    for (int e = 0; e < V; ++e) {
      in[e] = u32x4{0, 0, 0, 0};
      if (k0 + e < s.k) {
        const long long at = (long long)(k0 + e) * s.ldb + n0;
        if (at <= s.b_last) {
          in[e] = ld16_any(B + at);
        } else {
          T v[V];
#pragma unroll
          for (int u = 0; u < V; ++u) v[u] = n0 + u < s.n ? B[at + u] : T(0);
          __builtin_memcpy(&in[e], v, 16);
        }
      }
    }
    if constexpr (V == 8) {
      transpose8x8_b16(in, out);
    } else {
#pragma unroll
      for (int u = 0; u < 4; ++u) out[u] = u32x4{in[0][u], in[1][u], in[2][u], in[3][u]};
    }
#pragma unroll
    for (int u = 0; u < V; ++u)
      if (n0 + u < s.n) bp[(long long)(n0 + u) * chunks + kc] = out[u];
    return;
  }
  const uint32_t idx = (blockIdx.x - b_blocks) * convn::kThreads + threadIdx.x;
  const uint32_t m = fdiv(idx, s.div_chunks);
  if ((int)m >= s.m) return;
  const int k0 = (int)(idx - m * chunks) * V;
  const T* src = A + (long long)m * s.lda + k0;
  u32x4 out = {0, 0, 0, 0};
  if (k0 + V <= s.k) {
    out = ld16_any(src);
  } else if (k0 < s.k) {
    T v[V];
#pragma unroll
    for (int e = 0; e < V; ++e) v[e] = k0 + e < s.k ? src[e] : T(0);
    __builtin_memcpy(&out, v, 16);
  }
  ap[idx] = out;
}

// out[m][n] = round(sum over the splits of partial[split][m][n] + bias[n]), in split order; one
// wave per workgroup, as in gemm_splitk_reduce_kernel.
template <typename Tag>
__global__ __launch_bounds__(64) void gemm_packed_reduce_kernel(const float* __restrict__ partial, int splits,
                                                                typename convg::IgElem<Tag>::T* __restrict__ C,
                                                                const void* __restrict__ bias, int bias_kind, int M, int N,
                                                                long long ldc, FastDiv div_n) {
  using E = convg::IgElem<Tag>;
  using T = typename E::T;
  const uint32_t idx = blockIdx.x * 64 + threadIdx.x;
  const uint32_t m = fdiv(idx, div_n);
  if ((int)m >= M) return;
  const int n = (int)(idx - m * N);
  const long long plane = (long long)M * N;
  float v = partial[idx];
  for (int y = 1; y < splits; ++y) v += partial[y * plane + idx];
  if (bias_kind == 1) v += static_cast<const float*>(bias)[n];
  if (bias_kind == 2) v += E::to_float(static_cast<const T*>(bias)[n]);
  T* out = C + (long long)m * ldc + n;
  if constexpr (E::kPerChunk == 8) *out = (T)(Half16<Tag>::pack2(v, 0.f) & 0xffffu);
  else *out = v;
}

// The SIMT kernel's time follows K (one load latency per 32 of it), this form's two launches and
// the packing do not pay for less (us, this form / SIMT): 16-bit from 100 MFLOP or K = 500
// (1000x1501x1023: 19.5 / 151; 1x3692x523: 11.1 / 14.4; 250^3: 10.9 / 9.4; 8000x65x129: 12.0 / 16.1),
// fp32 from 200 MFLOP or K = 1000 (511x513x515: 16.9 / 30.3; 24x100x8000: 25 / 127; 1x3692x523:
// 16.9 / 10.8; 8000x65x129: 16.6 / 13.6), few fp32 rows against an rhs of over 32 MB or of very many
// columns not at all: the SIMT kernel then has its CUs' worth of tiles and reads rhs once
// (5x4313x7213: 238 / 149; 13x5900x1745: 68 / 38, but 4x8000x1000: 58 / 76; 46x10489x1809: 144 / 106,
// 36x9233x3429: 224 / 194, but 53x8945x2783: 148 / 160; 114x12697x2395: 264 / 242, but 108x12077x5391: 414 / 537).
inline bool gemm_packed_pays(long long M, long long N, long long K, bool f32) {
  if (f32 && M < 16 && (double)N * K > 8e6) return false;
  if (f32 && ((M <= 64 && N >= 9000) || (M <= 128 && N >= 12300))) return false;
  return K >= (f32 ? 1000 : 500) || 2.0 * M * N * K >= (f32 ? 2e8 : 1e8);
}

struct GemmPackedPlan {
  bool ok = false;
  long long m = 0, n = 0;  // rows of lhs and columns of rhs per piece
  int slices = 0;          // 128-byte K slices
  int bm = 64, ring = 5;   // tiles of bm columns x 64 rows
  int splits = 1, kcs = 0;
  size_t a_bytes = 0, b_bytes = 0, partial_bytes = 0;
  size_t bytes() const { return a_bytes + b_bytes + partial_bytes; }
};

inline GemmPackedPlan gemm_packed_plan(long long M, long long N, long long K, bool f32, long long max_bytes) {
  GemmPackedPlan p;
  const int es = f32 ? 4 : 2;
  const long long pitch = (K * es + 127) / 128 * 128;
  if (M < 1 || N < 1 || K < 1 || pitch * 512 > max_bytes) return p;
  // pieces of equal size whose packed rows fit three quarters of the workspace
  const long long rows = max_bytes / 4 * 3 / pitch;
  auto piece = [](long long extent, long long limit) {
    const long long count = (extent + limit - 1) / limit;
    return std::min(extent, ((extent + count - 1) / count + 127) / 128 * 128);
  };
  p.m = piece(M, std::max<long long>(128, rows / 2 / 128 * 128));
  p.n = piece(N, std::max<long long>(128, (rows - p.m) / 128 * 128));
  p.slices = (int)(pitch / 128);
  p.a_bytes = (size_t)(p.m * pitch);
  p.b_bytes = (size_t)(p.n * pitch);
  auto tiles = [&](int bm) { return ((p.n + bm - 1) / bm) * ((p.m + 63) / 64); };
  // tile and ring as for convolutions (conv_nhwc_plan)
  if (tiles(128) >= 512) {
    p.bm = 128;
    p.ring = p.slices <= 4 ? 2 : 3;
  } else {
    p.ring = tiles(64) > 512 ? 3 : 5;
  }
  // and split-K by the same time model
  const long long t = tiles(p.bm), mn = p.m * p.n, slice_ns = f32 ? 650 : 330;
  {
    long long best = 1, best_ns = (t + 511) / 512 * p.slices * slice_ns;
    for (long long sp = 2; sp <= p.slices / (f32 ? 4 : 8) && t * (sp - 1) < 512; ++sp) {
      const long long ns =
          (t * sp + 511) / 512 * ((p.slices + sp - 1) / sp) * slice_ns + sp * mn * 8 / 2000 + 4000;
      if (ns < best_ns) { best = sp; best_ns = ns; }
    }
    const int c = (int)((p.slices + best - 1) / best);
    const int splits = (p.slices + c - 1) / c;
    const size_t partial = (size_t)splits * mn * 4;
    if (splits > 1 && p.a_bytes + p.b_bytes + partial <= (size_t)max_bytes) {
      p.splits = splits;
      p.kcs = c;
      p.partial_bytes = partial;
    }
  }
  p.ok = true;
  return p;
}

// MFMA instructions of a matmul run by `plan` (16-bit: 16x16x32, fp32: 16x16x4).
inline long long gemm_packed_mfma(long long M, long long N, const GemmPackedPlan& plan, bool f32) {
  long long count = 0;
  for (long long m0 = 0; m0 < M; m0 += plan.m)
    for (long long n0 = 0; n0 < N; n0 += plan.n) {
      const long long tiles = (std::min(plan.n, N - n0) + plan.bm - 1) / plan.bm * ((std::min(plan.m, M - m0) + 63) / 64);
      count += tiles * plan.slices * (plan.bm / 16) * 4 * 2 * (f32 ? 4 : 1);
    }
  return count;
}

// bias_kind: 0 none, 1 fp32, 2 same dtype. Unit column strides; any row strides and alignment.
template <typename Tag>
hipError_t launch_gemm_packed(const void* A, const void* B, void* C, const void* bias, int bias_kind, int M, int N, int K,
                              long long lda, long long ldb, long long ldc, const GemmPackedPlan& plan, char* ws,
                              hipStream_t stream) {
  using T = typename convg::IgElem<Tag>::T;
  constexpr int V = convg::IgElem<Tag>::kPerChunk;
  constexpr int es = (int)sizeof(T);
  char* ap = ws;
  char* bp = ws + plan.a_bytes;
  float* partial = reinterpret_cast<float*>(ws + plan.a_bytes + plan.b_bytes);
  gemmx::Params s;
  s.k = K;
  s.lda = lda;
  s.ldb = ldb;
  s.pitch = (uint32_t)plan.slices * 128;
  s.div_chunks = make_fast_div(s.pitch / 16);
  convn::Geometry g = {};
  g.taps_w = 1;
  g.kh = g.kw = 1;
  g.cpr = (K + V - 1) / V;
  g.spr = plan.slices;
  g.hpr = 2 * plan.slices;
  g.slices = plan.slices;
  g.row_w = g.w_pitch = s.pitch;
  g.kcs = plan.splits > 1 ? plan.kcs : 0;
  g.div_spr = make_fast_div((uint32_t)g.spr);
  g.div_hpr = make_fast_div((uint32_t)g.hpr);
  g.div_taps_w = make_fast_div(1);
  g.bias_kind = bias_kind == 0 ? 0 : bias_kind + 2;  // per column
  for (long long m0 = 0; m0 < M; m0 += plan.m) {
    s.m = (int)std::min<long long>(plan.m, M - m0);
    for (long long n0 = 0; n0 < N; n0 += plan.n) {
      s.n = (int)std::min<long long>(plan.n, N - n0);
      s.b_last = (long long)(K - 1) * ldb + s.n - V;
      const long long b_threads = (long long)((s.n + V - 1) / V) * s.div_chunks.d;
      const long long a_threads = n0 == 0 ? (long long)s.m * s.div_chunks.d : 0;  // a piece of lhs is packed once
      const int b_blocks = (int)((b_threads + convn::kThreads - 1) / convn::kThreads);
      const int a_blocks = (int)((a_threads + convn::kThreads - 1) / convn::kThreads);
      hipLaunchKernelGGL((gemm_pack_kernel<Tag>), dim3(b_blocks + a_blocks), dim3(convn::kThreads), 0, stream,
                         static_cast<const T*>(A) + m0 * lda, static_cast<const T*>(B) + n0,
                         reinterpret_cast<u32x4*>(ap), reinterpret_cast<u32x4*>(bp), s, b_blocks);
      g.f = s.m;
      g.P = g.NP = s.n;
      g.x_bytes = (uint32_t)s.n * s.pitch;
      g.div_p = g.div_wo = make_fast_div((uint32_t)s.n);
      T* c = static_cast<T*>(C) + m0 * ldc + n0;
      g.out_pitch = (int)ldc;
      // stores of 8 or 4 columns where every row starts and ends on one (4: 8 bytes of 16-bit
      // values, 16 of fp32)
      const uintptr_t at = (uintptr_t)c;
      g.piece = es == 2 && s.n % 8 == 0 && ldc % 8 == 0 && at % 16 == 0 ? 8
                : s.n % 4 == 0 && ldc % 4 == 0 && at % (4 * es) == 0    ? 4
                                                                         : 1;
      const char* bsrc = bias == nullptr ? nullptr
                                         : static_cast<const char*>(bias) + n0 * (bias_kind == 1 ? 4 : es);
      launch_nhwc_gemm<Tag>(bp, ap, c, bsrc, g, plan.bm, plan.ring, plan.splits, partial, stream);
      if (plan.splits > 1)
        hipLaunchKernelGGL((gemm_packed_reduce_kernel<Tag>), dim3((unsigned)(((long long)s.m * s.n + 63) / 64)), dim3(64),
                           0, stream, partial, plan.splits, c, bsrc, bias_kind, s.m, s.n, ldc, make_fast_div((uint32_t)s.n));
      const hipError_t e = hipGetLastError();
      if (e != hipSuccess) return e;
    }
  }
  return hipGetLastError();
}

}  // namespace kg_gfx950
