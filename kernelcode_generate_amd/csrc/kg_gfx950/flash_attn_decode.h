// Attention with the keys of a (b,h) split over workgroups, queries in blocks of 16, fp32 online
// softmax, Q/K/V/O [B,H,S,D]: 16-bit calls of few queries with D = 64 or 128 (a decoding step; no
// mask), 16-bit calls of other head dims (multiples of 8, causal or not), and fp32 calls
// (fa_split_f32_kernel below).
//
// A decoding step reads K and V once and does little else, so what bounds it is how much of the
// chip keeps loads in flight. fa_fwd_mfma_kernel gives a (b,h) one workgroup (B H = 128: half
// the CUs, 3.4 TB/s) whose K/V tiles wait for each other at barriers; here a (b,h)'s keys are
// split over workgroups until there are two per CU, and each wave walks its own steps of keys
// with its own running max and sums, its next step's K and V (16 KiB) in flight in registers
// during the current one: no LDS, no barrier until the end.
//
// A step is kNC chunks of 32 keys. S^T = K Q^T as in flash_attn_mfma.h (v_mfma_f32_16x16x32,
// operand A 16 keys x 32 d straight from K's rows, operand B Q^T in registers): lane l holds
// the scores of query l%16 against keys 16kb + 4(l/16) + 0..3. O^T += V^T P^T contracts a chunk
// in the key order a lane row holds P in, so lane row r needs V of keys 4r + 0..3 and 16 + 4r +
// 0..3: it loads those 8 rows, D/16 columns per lane (whole rows per 16 lanes), and
// transposes them in registers; block c of O^T is then rows d = (D/16) x + c, x = 0..15.
// The waves' and then the splits' results (m, l, O) are combined as the online softmax does.
#pragma once

#include "common.h"
#include "conv2d_igemm.h"
#include "flash_attn.h"
#include "flash_attn_mfma.h"

namespace kg_gfx950 {

namespace fad {
constexpr int kWaves = 4;
constexpr int kThreads = 64 * kWaves;
constexpr int kMaxQ = 16;
template <int D>
constexpr int step_keys() { return D == 128 ? 32 : 64; }  // 16 KiB of K and V
// The lowest running max: a score of -inf (infinite inputs) has weight 0 beside finite ones,
// also where a whole step has no other.
constexpr float kMinMax = -3.0e38f;

// O^T += V^T P^T in fp32 over the 4 NG keys of a step: MFMA n contracts keys key0 + 16 (n/4) +
// 4 (l/16) + n%4, of which this lane holds query l16's weight p[n] and V's values v(n, e) of block e.
// masked: the step has keys that some of the queries q0 + 0..15 do not see (their weights are 0). A
// weight of 0 does not take an infinity or NaN out of the sum, so where such a step holds one,
// every query gets a pass of its own with zeros in place of the keys after it. Finite values (a test of
// V's registers in one step per block of queries) take the one pass.
// non_finite() tests this lane's: on the stored words, as the widened values of a whole step, kept from the
// test for the products, spilled 256 registers (bf16 16x389x389x80 17 -> 40 us).
template <int NE, int NG, typename Values, typename Test>
__device__ __forceinline__ void add_pv_f32(f32x4 (&o)[NE], const float (&p)[NG], Values v, Test non_finite, bool masked,
                                           int key0, int q0, int l16, int lr) {
  bool apart = false;
  if (masked) apart = __builtin_amdgcn_ballot_w64(non_finite()) != 0;
  if (!apart) {
#pragma unroll
    for (int n = 0; n < NG; ++n)
#pragma unroll
      for (int e = 0; e < NE; ++e) o[e] = __builtin_amdgcn_mfma_f32_16x16x4f32(v(n, e), p[n], o[e], 0, 0, 0);
    return;
  }
#pragma unroll
  for (int e = 0; e < NE; ++e) {
    f32x4 sum = o[e];
#pragma unroll 1
    for (int q = 0; q < kMaxQ; ++q) {
      f32x4 t = o[e];
#pragma unroll
      for (int n = 0; n < NG; ++n) {
        const float seen = key0 + 16 * (n >> 2) + 4 * lr + (n & 3) <= q0 + q ? v(n, e) : 0.f;
        t = __builtin_amdgcn_mfma_f32_16x16x4f32(seen, p[n], t, 0, 0, 0);
      }
      if (l16 == q) sum = t;
    }
    o[e] = sum;
  }
}
}  // namespace fad

// splits == 1: O is written; else partial[(bh splits + split) s_q + q][D + 2] takes O (not
// normalised), m (log2 units) and l.
// kAny: head dims d < D (multiples of 8, rows padded with zeros in registers), causal or not. No tiled
// kernel has these dims, and the SIMT kernel keeps its probabilities in fp32: so does this form,
// whose P V and row sums are fp32 products (v_mfma_f32_16x16x4_f32). They take sixteen times the
// MFMA time of the 16-bit ones and bound it.
template <typename Tag, int D, bool kAny>
__global__ __launch_bounds__(fad::kThreads, 2) void fa_decode_kernel(const uint16_t* __restrict__ Q,
                                                                     const uint16_t* __restrict__ K,
                                                                     const uint16_t* __restrict__ V,
                                                                     uint16_t* __restrict__ O, int s_q, int s_kv, int d_any,
                                                                     int causal, float scale_log2, int splits, int split_keys,
                                                                     float* __restrict__ partial) {
  using namespace fad;
  using H = Half16<Tag>;
  constexpr int NDS = D / 32;            // 32-deep d steps of S^T
  constexpr int NE = D / 16;             // V columns per lane: blocks of O^T
  constexpr int kStep = step_keys<D>();
  constexpr int NC = kStep / 32;         // 32-key chunks per step
  using VRow = typename std::conditional<NE == 8, u32x4, u32x2>::type;
  struct Buf {
    u32x4 k[2 * NC][NDS];
    VRow v[NC][8];
  };
  __shared__ float o_lds[kWaves][kMaxQ][D];
  __shared__ float ml_lds[kWaves][kMaxQ][2];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, lr = lane >> 4;
  const int bh = blockIdx.x / splits, split = blockIdx.x - bh * splits;
  const int q0 = blockIdx.y * kMaxQ, nq = min(s_q - q0, kMaxQ);  // this workgroup's queries
  const int d_row = kAny ? d_any : D;
  const bool diagonal = kAny && causal != 0;
  const int key_lo = split * split_keys;
  const int key_hi = min(diagonal ? min(s_kv, q0 + nq) : s_kv, key_lo + split_keys);
  const uint16_t* Kb = K + (long long)bh * s_kv * d_row;
  const uint16_t* Vb = V + (long long)bh * s_kv * d_row;

  u32x4 qf[NDS];
#pragma unroll
  for (int s = 0; s < NDS; ++s)
    qf[s] = l16 < nq && (!kAny || 32 * s + 8 * lr < d_row)
                ? ld16(Q + ((long long)bh * s_q + q0 + l16) * d_row + 32 * s + 8 * lr)
                : u32x4{0, 0, 0, 0};

  // keys past key_hi (the last step of a range): rows of zeros
  auto load = [&](Buf& b, int key0, bool whole) __attribute__((always_inline)) {
#pragma unroll
    for (int kb = 0; kb < 2 * NC; ++kb) {
      const int key = key0 + 16 * kb + l16;
      const uint16_t* row = Kb + (long long)key * d_row + 8 * lr;
#pragma unroll
      for (int s = 0; s < NDS; ++s)
        b.k[kb][s] = (whole || key < key_hi) && (!kAny || 32 * s + 8 * lr < d_row) ? ld16(row + 32 * s)
                                                                                   : u32x4{0, 0, 0, 0};
    }
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int r = 0; r < 8; ++r) {
        const int key = key0 + 32 * c + 4 * lr + (r < 4 ? r : 12 + r);
        b.v[c][r] = (whole || key < key_hi) && (!kAny || NE * l16 < d_row)
                        ? *reinterpret_cast<const VRow*>(Vb + (long long)key * d_row + NE * l16)
                        : VRow{};
      }
  };

  f32x4 o[NE];
#pragma unroll
  for (int c = 0; c < NE; ++c) o[c] = f32x4{0.f, 0.f, 0.f, 0.f};
  f32x4 l_run = {0.f, 0.f, 0.f, 0.f};
  float m_run = kMinMax;
  const u32x4 ones = {H::kOnePair, H::kOnePair, H::kOnePair, H::kOnePair};

  auto compute = [&](Buf& b, int key0, bool whole) __attribute__((always_inline)) {
    f32x4 sc[2 * NC];
#pragma unroll
    for (int kb = 0; kb < 2 * NC; ++kb) {
      sc[kb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < NDS; ++s) sc[kb] = H::mfma16(b.k[kb][s], qf[s], sc[kb]);
    }
    if (!whole || (diagonal && key0 + kStep - 1 > q0)) {
      const int last = diagonal ? min(key_hi - 1, q0 + l16) : key_hi - 1;  // this query's last key
#pragma unroll
      for (int kb = 0; kb < 2 * NC; ++kb)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (key0 + 16 * kb + 4 * lr + i > last) sc[kb][i] = -INFINITY;
    }
    float mx = sc[0][0];
#pragma unroll
    for (int x = 1; x < 8 * NC; ++x) mx = __builtin_elementwise_maximum(mx, (float)sc[x >> 2][x & 3]);
    float mx2 = mx;
    fa::rows4_combine<true>(mx, mx2);
    const float m_new = __builtin_elementwise_maximum(m_run, mx * scale_log2);
    if (__builtin_amdgcn_ballot_w64(m_new > m_run || m_new != m_new)) {
      const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
      m_run = m_new;
      l_run *= alpha;
#pragma unroll
      for (int c = 0; c < NE; ++c) o[c] *= alpha;
    }
    if constexpr (kAny) {
      // P stays fp32 and V's elements are widened
      float p[8 * NC];
#pragma unroll
      for (int n = 0; n < 8 * NC; ++n) {
        p[n] = __builtin_amdgcn_exp2f(__builtin_fmaf((float)sc[n >> 2][n & 3], scale_log2, -m_run));
        l_run[0] += p[n];
      }
      auto value = [&](int n, int e) __attribute__((always_inline)) {  // key 16 (n/4) + 4 (l/16) + n%4 of the step
        const uint32_t pair = b.v[n >> 3][n & 7][e >> 1];
        return H::to_float((e & 1) ? pair >> 16 : pair & 0xffffu);
      };
      auto non_finite = [&]() __attribute__((always_inline)) {  // an exponent of ones carries into its sign bit
        uint32_t carry = 0;
#pragma unroll
        for (int r = 0; r < 8 * NC; ++r)
#pragma unroll
          for (int w = 0; w < NE / 2; ++w) carry |= (b.v[r >> 3][r & 7][w] & H::kExpPair) + H::kExpUnitPair;
        return (carry & 0x80008000u) != 0;
      };
      add_pv_f32(o, p, value, non_finite, diagonal && key0 + kStep - 1 > q0, key0, q0, l16, lr);
    } else {
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        u32x4 pp;  // keys 32c + 4 lr + 0..3, then + 16
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int q = 0; q < 2; ++q) {
            const float p0 = __builtin_amdgcn_exp2f(__builtin_fmaf(sc[2 * c + h][2 * q], scale_log2, -m_run));
            const float p1 = __builtin_amdgcn_exp2f(__builtin_fmaf(sc[2 * c + h][2 * q + 1], scale_log2, -m_run));
            pp[2 * h + q] = H::pack2(p0, p1);
          }
#pragma unroll
        for (int e = 0; e < NE; ++e) {  // column e of each lane's 8 rows
          u32x4 vt;
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const uint32_t x = b.v[c][2 * q][e >> 1], y = b.v[c][2 * q + 1][e >> 1];
            vt[q] = (e & 1) ? hi_halves(x, y) : lo_halves(x, y);
          }
          o[e] = H::mfma16(vt, pp, o[e]);
        }
        l_run = H::mfma16(ones, pp, l_run);
      }
    }
  };

  // this wave's steps: key_lo + kStep (wave + 4 i); all but the range's last are whole
  constexpr int kStride = kStep * kWaves;
  int key = key_lo + kStep * wave;
  Buf b0, b1;
  if (key + kStep <= key_hi) {
    load(b0, key, true);
    for (;;) {
      const bool more1 = key + kStride + kStep <= key_hi;
      if (more1) load(b1, key + kStride, true);
      __builtin_amdgcn_sched_barrier(0);
      compute(b0, key, true);
      key += kStride;
      if (!more1) break;
      const bool more0 = key + kStride + kStep <= key_hi;
      if (more0) load(b0, key + kStride, true);
      __builtin_amdgcn_sched_barrier(0);
      compute(b1, key, true);
      key += kStride;
      if (!more0) break;
    }
  }
  if (key < key_hi) {
    load(b0, key, false);
    compute(b0, key, false);
  }

  // ---- combine the waves (kAny: first the four lane rows' keys of the row sum) ----
  if constexpr (kAny) {
    float l0 = l_run[0], l1 = l0;
    fa::rows4_combine<false>(l0, l1);
    l_run[0] = l0;
  }
  if (l16 < nq) {
#pragma unroll
    for (int e = 0; e < NE; ++e)
#pragma unroll
      for (int i = 0; i < 4; ++i) o_lds[wave][l16][NE * (4 * lr + i) + e] = o[e][i];
    if (lr == 0) {
      ml_lds[wave][l16][0] = m_run;
      ml_lds[wave][l16][1] = l_run[0];
    }
  }
  __syncthreads();
  for (int x = tid; x < nq * (D / 2); x += kThreads) {
    const int q = x / (D / 2), d = 2 * (x % (D / 2));
    if (kAny && d >= d_row) continue;
    float m = ml_lds[0][q][0];
#pragma unroll
    for (int w = 1; w < kWaves; ++w) m = __builtin_elementwise_maximum(m, ml_lds[w][q][0]);
    float l = 0.f, o0 = 0.f, o1 = 0.f;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      const float a = __builtin_amdgcn_exp2f(ml_lds[w][q][0] - m);
      l += a * ml_lds[w][q][1];
      o0 += a * o_lds[w][q][d];
      o1 += a * o_lds[w][q][d + 1];
    }
    if (splits == 1) {
      const float inv = 1.f / l;
      *reinterpret_cast<uint32_t*>(O + ((long long)bh * s_q + q0 + q) * d_row + d) = H::pack2(o0 * inv, o1 * inv);
    } else {
      float* p = partial + ((long long)blockIdx.x * s_q + q0 + q) * (D + 2);
      *reinterpret_cast<f32x2*>(p + d) = f32x2{o0, o1};
      if (d == 0) *reinterpret_cast<f32x2*>(p + D) = f32x2{m, l};
    }
  }
}

// One wave per (b,h) and query: the splits' partials combined and normalised, D / 64 columns per lane.
template <typename Tag, int D>
__global__ __launch_bounds__(64) void fa_decode_combine_kernel(const float* __restrict__ partial,
                                                               typename convg::IgElem<Tag>::T* __restrict__ O, int s_q,
                                                               int d_row, int splits) {
  const int lane = threadIdx.x;
  const int bh = blockIdx.x / s_q, q = blockIdx.x - bh * s_q;
  const float* p = partial + ((long long)bh * splits * s_q + q) * (D + 2);
  const long long pitch = (long long)s_q * (D + 2);
  float m = -INFINITY;
  for (int s = lane; s < splits; s += 64) m = fmaxf(m, p[s * pitch + D]);
  m = wave_max(m);
  float l = 0.f, o[D / 64];
#pragma unroll
  for (int e = 0; e < D / 64; ++e) o[e] = 0.f;
#pragma unroll 8
  for (int s = 0; s < splits; ++s) {
    const float a = __builtin_amdgcn_exp2f(p[s * pitch + D] - m);
    l += a * p[s * pitch + D + 1];
#pragma unroll
    for (int e = 0; e < D / 64; ++e) o[e] += a * p[s * pitch + lane + 64 * e];
  }
  const float inv = 1.f / l;
#pragma unroll
  for (int e = 0; e < D / 64; ++e) {
    const int d = lane + 64 * e;
    if (d >= d_row) continue;
    auto* out = O + ((long long)bh * s_q + q) * d_row + d;
    if constexpr (convg::IgElem<Tag>::kPerChunk == 8) *out = (uint16_t)(Half16<Tag>::pack2(o[e] * inv, 0.f) & 0xffffu);
    else *out = o[e] * inv;
  }
}

// fp32 form (v_mfma_f32_16x16x4_f32, one k per lane), any head dim d <= 16 NE that is a multiple
// of 4, causal or not: a step is 16 keys; S^T takes 16 d in four MFMAs from 16-byte pieces of K's
// rows (element j of every lane's piece), O^T takes the keys 4(l/16) + i of a step in MFMA i
// against V[key][16 e + l%16], which needs no transpose. fa_fwd_simt_kernel, one workgroup per
// query, read every key row once per query and lane: 16x389x389x80 took 133 us.
template <int NE>
__global__ __launch_bounds__(fad::kThreads, 2) void fa_split_f32_kernel(const float* __restrict__ Q,
                                                                        const float* __restrict__ K,
                                                                        const float* __restrict__ V,
                                                                        float* __restrict__ O, int s_q, int s_kv, int d_row,
                                                                        int causal, float scale_log2, int splits,
                                                                        int split_keys, float* __restrict__ partial) {
  using namespace fad;
  constexpr int D = NE <= 4 ? 64 : 128;  // columns of a partial row
  constexpr int kStep = 16;
  struct Buf {
    f32x4 k[NE];
    float v[4][NE];
  };
  __shared__ float o_lds[kWaves][kMaxQ][16 * NE + 1];
  __shared__ float ml_lds[kWaves][kMaxQ][2];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, lr = lane >> 4;
  const int bh = blockIdx.x / splits, split = blockIdx.x - bh * splits;
  const int q0 = blockIdx.y * kMaxQ, nq = min(s_q - q0, kMaxQ);
  const int key_lo = split * split_keys;
  const int key_hi = min(causal ? min(s_kv, q0 + nq) : s_kv, key_lo + split_keys);
  const float* Kb = K + (long long)bh * s_kv * d_row;
  const float* Vb = V + (long long)bh * s_kv * d_row;
  const f32x4 zero4 = {0.f, 0.f, 0.f, 0.f};

  f32x4 qf[NE];
#pragma unroll
  for (int s = 0; s < NE; ++s)
    qf[s] = l16 < nq && 16 * s + 4 * lr < d_row
                ? *reinterpret_cast<const f32x4*>(Q + ((long long)bh * s_q + q0 + l16) * d_row + 16 * s + 4 * lr)
                : zero4;

  auto load = [&](Buf& b, int key0) __attribute__((always_inline)) {
    const int kk = key0 + l16;
#pragma unroll
    for (int s = 0; s < NE; ++s)
      b.k[s] = kk < key_hi && 16 * s + 4 * lr < d_row
                   ? *reinterpret_cast<const f32x4*>(Kb + (long long)kk * d_row + 16 * s + 4 * lr)
                   : zero4;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int key = key0 + 4 * lr + i;
#pragma unroll
      for (int e = 0; e < NE; ++e)
        b.v[i][e] = key < key_hi && 16 * e + l16 < d_row ? Vb[(long long)key * d_row + 16 * e + l16] : 0.f;
    }
  };

  f32x4 o[NE];
#pragma unroll
  for (int e = 0; e < NE; ++e) o[e] = zero4;
  float l_run = 0.f;  // this lane's keys' share of the row sum
  float m_run = kMinMax;
  auto compute = [&](Buf& b, int key0) __attribute__((always_inline)) {
    // two accumulators: half as long a chain of dependent MFMAs
    f32x4 sc = zero4, sd = zero4;
#pragma unroll
    for (int s = 0; s < NE; ++s)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        f32x4& acc = j & 1 ? sd : sc;
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32((float)b.k[s][j], (float)qf[s][j], acc, 0, 0, 0);
      }
#pragma unroll
    for (int i = 0; i < 4; ++i) sc[i] += sd[i];
    const int last = causal ? min(key_hi - 1, q0 + l16) : key_hi - 1;  // this query's last key
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (key0 + 4 * lr + i > last) sc[i] = -INFINITY;
    float mx = __builtin_elementwise_maximum(__builtin_elementwise_maximum((float)sc[0], (float)sc[1]),
                                             __builtin_elementwise_maximum((float)sc[2], (float)sc[3]));
    float mx2 = mx;
    fa::rows4_combine<true>(mx, mx2);
    const float m_new = __builtin_elementwise_maximum(m_run, mx * scale_log2);
    if (__builtin_amdgcn_ballot_w64(m_new > m_run || m_new != m_new)) {
      const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
      m_run = m_new;
      l_run *= alpha;
#pragma unroll
      for (int e = 0; e < NE; ++e) o[e] *= alpha;
    }
    float p[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      p[i] = __builtin_amdgcn_exp2f(__builtin_fmaf((float)sc[i], scale_log2, -m_run));
      l_run += p[i];
    }
    auto value = [&](int n, int e) __attribute__((always_inline)) { return b.v[n][e]; };
    auto non_finite = [&]() __attribute__((always_inline)) {
      bool any = false;
#pragma unroll
      for (int n = 0; n < 4; ++n)
#pragma unroll
        for (int e = 0; e < NE; ++e) any |= !__builtin_isfinite(b.v[n][e]);
      return any;
    };
    add_pv_f32(o, p, value, non_finite, causal != 0 && key0 + kStep - 1 > q0, key0, q0, l16, lr);
  };

  constexpr int kStride = kStep * kWaves;
  Buf b0, b1;
  int key = key_lo + kStep * wave;
  if (key < key_hi) {
    load(b0, key);
    for (;;) {
      const bool more1 = key + kStride < key_hi;
      if (more1) load(b1, key + kStride);
      __builtin_amdgcn_sched_barrier(0);
      compute(b0, key);
      key += kStride;
      if (!more1) break;
      const bool more0 = key + kStride < key_hi;
      if (more0) load(b0, key + kStride);
      __builtin_amdgcn_sched_barrier(0);
      compute(b1, key);
      key += kStride;
      if (!more0) break;
    }
  }

  // the four lane rows' row sums, then the waves
  float l2 = l_run;
  fa::rows4_combine<false>(l_run, l2);
  if (l16 < nq) {
#pragma unroll
    for (int e = 0; e < NE; ++e)
#pragma unroll
      for (int i = 0; i < 4; ++i) o_lds[wave][l16][16 * e + 4 * lr + i] = o[e][i];
    if (lr == 0) {
      ml_lds[wave][l16][0] = m_run;
      ml_lds[wave][l16][1] = l_run;
    }
  }
  __syncthreads();
  for (int x = tid; x < nq * 16 * NE; x += kThreads) {
    const int q = x / (16 * NE), d = x % (16 * NE);
    if (d >= d_row) continue;
    float m = ml_lds[0][q][0];
#pragma unroll
    for (int w = 1; w < kWaves; ++w) m = __builtin_elementwise_maximum(m, ml_lds[w][q][0]);
    float l = 0.f, ov = 0.f;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      const float a = __builtin_amdgcn_exp2f(ml_lds[w][q][0] - m);
      l += a * ml_lds[w][q][1];
      ov += a * o_lds[w][q][d];
    }
    if (splits == 1) {
      O[((long long)bh * s_q + q0 + q) * d_row + d] = ov / l;
    } else {
      float* p = partial + ((long long)blockIdx.x * s_q + q0 + q) * (D + 2);
      p[d] = ov;
      if (d == 0) {
        p[D] = m;
        p[D + 1] = l;
      }
    }
  }
}

// The calls it takes: up to 16 queries always; more, in blocks of 16 that each read the keys
// again, while the blocks are few beside the 512 workgroups that fill the chip and the keys many
// (us, this kernel / fa_fwd_mfma_kernel, bf16, B H x S_q x S_kv x D: 128x1x4096x128 44 / 81,
// 8x1x16384x128 17 / 298, 8x64x16384x128 30 / 299, 8x128x1024x128 14.6 / 19.2, 128x17x2048x128 (256
// blocks) 43 / 43, 32x128x4096x128 (256 blocks) 47 / 64, 256x17x1000x128 (512 blocks) 38 / 32).
inline int fa_decode_blocks(const FaShape& s) { return (s.s_q + fad::kMaxQ - 1) / fad::kMaxQ; }
inline bool fa_decode_supported(const FaShape& s) {
  const long long blocks = (long long)s.bh * fa_decode_blocks(s);
  const bool pays = s.s_q <= fad::kMaxQ ||
                    (s.s_kv >= 1024 && (blocks <= 128 || (blocks <= 256 && s.s_q >= 64 && s.s_kv >= 2048)));
  return s.s_q >= 1 && s.s_kv >= 1 && !s.causal && (s.d == 64 || s.d == 128) && s.scale > 0.f && s.bh >= 1 &&
         s.bh <= (1 << 20) && pays;
}
// Head dims the tiled kernels do not have, which otherwise run one workgroup per query (16-bit:
// multiples of 8 from 24, fp32: of 4; causal or not), any call (us, this kernel /
// fa_fwd_simt_kernel: 16x389x389x80 fp32 24 / 131, bf16 16.9 / 102; 128x512x512x96 causal bf16 81 /
// 779; 32x1x2048x96 bf16 11.2 / 103). Below 24 the padding to 64 is most of the work. And fp32 with D = 64 or 128, causal or not, of up
// to 16 queries or 512 blocks of them, where fa_fwd_f32_mfma_kernel's blocks of 128 queries leave
// CUs idle (8x1x8192x128 23 / 1179; 16x512x512x64 22 / 47; 24x64x64x64 10.5 / 9.5, x128 10.7 / 13.5;
// 256x64x64x64, 1024 blocks, 11.9 / 9.4; 32x1024x1024x64, 2048 blocks, 151 / 95).
inline bool fa_split_supported(const FaShape& s, bool f32) {
  if (!(s.s_q >= 1 && s.s_kv >= 1 && s.scale > 0.f && s.bh >= 1 && s.bh <= (1 << 20) && fa_decode_blocks(s) <= 65535))
    return false;
  if (s.d != 64 && s.d != 128) return s.d >= 24 && s.d <= 128 && s.d % (f32 ? 4 : 8) == 0;
  if (f32) return s.s_q <= fad::kMaxQ || (long long)s.bh * fa_decode_blocks(s) <= 512;
  return fa_decode_supported(s);
}

// Splits of a call's keys (ranges of whole steps): two workgroups per CU of the MI355X (256),
// each wave with at least two steps. splits == 1 needs no workspace.
struct FaDecodePlan {
  int splits, split_keys;
  size_t bytes;  // of partials
};
inline FaDecodePlan fa_decode_plan(const FaShape& s, bool f32, bool may_split) {
  const int step = f32 ? 16 : s.d > 64 ? fad::step_keys<128>() : fad::step_keys<64>();
  const int cols = s.d > 64 ? 128 : 64;
  const long long rounds = ((long long)s.s_kv + step * fad::kWaves - 1) / (step * fad::kWaves);  // steps per wave in all
  long long splits = std::min<long long>(512 / ((long long)s.bh * fa_decode_blocks(s)), rounds / 2);
  if (splits < 2 || !may_split) return FaDecodePlan{1, s.s_kv, 0};
  const long long per = (rounds + splits - 1) / splits;
  splits = (rounds + per - 1) / per;
  return FaDecodePlan{(int)splits, (int)(per * step * fad::kWaves),
                      splits > 1 ? (size_t)s.bh * splits * s.s_q * (cols + 2) * sizeof(float) : 0};
}
// 16-bit calls of the kAny form (D = 64 and 128 come here without a mask only).
inline bool fa_decode_any(const FaShape& s) { return s.causal || (s.d != 64 && s.d != 128); }

// MFMA instructions: per step and block of queries 2 S^T blocks x D/32 and D/16 + 1 for O^T and the
// row sums per 32 keys (other head dims: 8 fp32 ones x D/16 for O^T, counted apart); fp32 4 for S^T
// and 4 for O^T per 16 d and 16 keys. Causal blocks stop at their last query's step.
struct FaDecodeMfma {
  long long h16, f32;  // v_mfma_f32_16x16x32 (16 cycles), v_mfma_f32_16x16x4_f32 (32 cycles)
};
inline FaDecodeMfma fa_decode_mfma(const FaShape& s, bool f32, const FaDecodePlan& plan) {
  const int step = f32 ? 16 : s.d > 64 ? fad::step_keys<128>() : fad::step_keys<64>();
  const int D = s.d > 64 ? 128 : 64, NE = s.d <= 64 ? 4 : s.d <= 96 ? 6 : 8;
  long long steps = 0;
  for (int b = 0; b < fa_decode_blocks(s); ++b) {
    const int end = s.causal ? std::min(s.s_kv, std::min((b + 1) * fad::kMaxQ, s.s_q)) : s.s_kv;
    for (long long lo = 0; lo < end; lo += plan.split_keys)
      steps += (std::min<long long>(plan.split_keys, end - lo) + step - 1) / step;
  }
  const long long chunks = s.bh * steps * (step / 32);
  if (f32) return FaDecodeMfma{0, s.bh * steps * 8 * NE};
  if (fa_decode_any(s)) return FaDecodeMfma{chunks * (D / 16), chunks * 8 * (D / 16)};
  return FaDecodeMfma{chunks * (D / 16 + D / 16 + 1), 0};
}

template <typename Tag, int D, bool kAny>
hipError_t launch_fa_decode_d(const uint16_t* q, const uint16_t* k, const uint16_t* v, uint16_t* o, const FaShape& s,
                              const FaDecodePlan& plan, float* partial, hipStream_t stream) {
  hipLaunchKernelGGL((fa_decode_kernel<Tag, D, kAny>), dim3(s.bh * plan.splits, fa_decode_blocks(s)),
                     dim3(fad::kThreads), 0, stream, q, k, v, o, s.s_q, s.s_kv, s.d, s.causal,
                     s.scale * 1.4426950408889634f, plan.splits, plan.split_keys, partial);
  if (plan.splits > 1)
    hipLaunchKernelGGL((fa_decode_combine_kernel<Tag, D>), dim3(s.bh * s.s_q), dim3(64), 0, stream, partial, o, s.s_q,
                       s.d, plan.splits);
  return hipGetLastError();
}

template <typename Tag>
hipError_t launch_fa_decode(const uint16_t* q, const uint16_t* k, const uint16_t* v, uint16_t* o, const FaShape& s,
                            const FaDecodePlan& plan, float* partial, hipStream_t stream) {
  if (fa_decode_any(s)) {
    if (s.d > 64) return launch_fa_decode_d<Tag, 128, true>(q, k, v, o, s, plan, partial, stream);
    return launch_fa_decode_d<Tag, 64, true>(q, k, v, o, s, plan, partial, stream);
  }
  if (s.d == 128) return launch_fa_decode_d<Tag, 128, false>(q, k, v, o, s, plan, partial, stream);
  return launch_fa_decode_d<Tag, 64, false>(q, k, v, o, s, plan, partial, stream);
}

template <int NE>
void launch_fa_split_f32_ne(const float* q, const float* k, const float* v, float* o, const FaShape& s,
                            const FaDecodePlan& plan, float* partial, hipStream_t stream) {
  hipLaunchKernelGGL((fa_split_f32_kernel<NE>), dim3(s.bh * plan.splits, fa_decode_blocks(s)), dim3(fad::kThreads), 0,
                     stream, q, k, v, o, s.s_q, s.s_kv, s.d, s.causal, s.scale * 1.4426950408889634f, plan.splits,
                     plan.split_keys, partial);
}
template <typename Tag>
hipError_t launch_fa_split_f32(const float* q, const float* k, const float* v, float* o, const FaShape& s,
                               const FaDecodePlan& plan, float* partial, hipStream_t stream) {
  if (s.d <= 64) launch_fa_split_f32_ne<4>(q, k, v, o, s, plan, partial, stream);
  else if (s.d <= 96) launch_fa_split_f32_ne<6>(q, k, v, o, s, plan, partial, stream);
  else launch_fa_split_f32_ne<8>(q, k, v, o, s, plan, partial, stream);
  if (plan.splits > 1) {
    if (s.d <= 64)
      hipLaunchKernelGGL((fa_decode_combine_kernel<Tag, 64>), dim3(s.bh * s.s_q), dim3(64), 0, stream, partial, o, s.s_q,
                         s.d, plan.splits);
    else
      hipLaunchKernelGGL((fa_decode_combine_kernel<Tag, 128>), dim3(s.bh * s.s_q), dim3(64), 0, stream, partial, o,
                         s.s_q, s.d, plan.splits);
  }
  return hipGetLastError();
}

}  // namespace kg_gfx950
