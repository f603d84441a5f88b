// gemm_mid_kernel: bf16/f16 GEMM in 128 x 128 tiles, for outputs of too few 128 x 256 tiles to
// give every CU one (2048^3: 128 of those, 26 us, half the chip idle; 256 of these, 18 us). Any M;
// N and K multiples of 8 (as gemm_pipe_kernel).
//
// Four waves, one per SIMD, each a 64 x 64 quarter (4 x 4 blocks of v_mfma_f32_16x16x32). K goes
// in slices of 64, two steps of 32: a step's 16 MFMAs run from registers while the next step's
// 8 fragments are read from LDS and 4 of the wave's 8 copies of a later slice are issued. With
// 16 MFMAs a step, a barrier per step would cost a fifth of it, hence 64-deep slices and one
// barrier per two steps: the barrier before a slice's second step finds all its fragments read,
// so it both publishes the next slice's copies and frees this slice's stage for its refill.
// kStages = 4 (128 KiB of LDS) where each CU has one workgroup, 2 (64 KiB, two workgroups per
// CU, one's MFMAs under the other's waits) for larger grids.
//
// LDS: lhs rows of 128 bytes ([m][64 k]), chunk c of row r at c ^ ((r >> 1) & 7); rhs rows of 256
// bytes ([k][128 n]), chunk c of row k at c ^ b_mask(k), read with ds_read_b64_tr_b16 as in
// gemm_pipe_kernel. Both patterns hit distinct banks. Each output sums its 32-deep MFMAs in k
// order, as the other 16-bit kernels do: the same bits.
#pragma once

#include "common.h"
#include "gemm.h"
#include "lds_dma.h"

namespace kg_gfx950 {

namespace gemmm {
constexpr int kT = 128;    // tile rows and columns
constexpr int kBK = 64;    // K slice
constexpr int kThreads = 256;
constexpr int kOperand = kT * kBK * 2;  // bytes of one operand's stage
__device__ __forceinline__ int a_swz(int row) { return (row >> 1) & 7; }
}  // namespace gemmm

// kRagged: M % 128, N % 128 or K % 64 non-zero: copies through buffer loads that land zeros
// outside the matrices, and stores only inside.
template <typename Tag, int kBias, int kStages, bool kRagged>
__global__ __launch_bounds__(gemmm::kThreads, kStages == 2 ? 2 : 1) void gemm_mid_kernel(
    const uint16_t* __restrict__ A, const uint16_t* __restrict__ B, uint16_t* __restrict__ C,
    const void* __restrict__ bias, int M, int N, int K, long long lda, long long ldb, long long ldc) {
  using namespace gemmm;
  using gemmp::b_mask;
  using H = Half16<Tag>;
  constexpr int kPieces = 8;  // copies per wave and slice: 4 lhs (8 rows each), 4 rhs (4 k-rows each)
  __shared__ __attribute__((aligned(1024))) char lds[kStages * 2 * kOperand];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  const int tiles_n = (N + kT - 1) / kT, tiles_m = (M + kT - 1) / kT;
  // each XCD takes a contiguous range of tiles in groups of 4 tile rows (few panels per L2)
  const int total = gridDim.x, xcd = blockIdx.x % 8;
  const int logical = xcd * (total / 8) + min(xcd, total % 8) + blockIdx.x / 8;
  constexpr int kGroupM = 4;
  const int group = logical / (kGroupM * tiles_n);
  const int first_m = group * kGroupM;
  const int gm = min(tiles_m - first_m, kGroupM);
  const int in_group = logical - group * kGroupM * tiles_n;
  const int m0 = (first_m + in_group % gm) * kT;
  const int n0 = (in_group / gm) * kT;

  // ---- HBM -> LDS copies. lhs piece p: rows (wave*4 + p)*8 + lane/8, slot lane%8; a_swz of those
  // rows depends on the lane and p's parity. rhs piece p: k-rows (wave*4 + p)*4 + lane/16, slot
  // lane%16; b_mask depends on the lane and p/2 ----
  uint32_t a_off[4], b_off[4];
  int a_k[2];  // a lane's k within the slice, by p's parity
#pragma unroll
  for (int p = 0; p < 4; ++p) {
    const int row = (wave * 4 + p) * 8 + (lane >> 3);
    const int c = (lane & 7) ^ a_swz(row);
    a_off[p] = (uint32_t)((row * lda + 8 * c) * 2);
    a_k[p & 1] = 8 * c;
    if (kRagged && m0 + row >= M) a_off[p] = kBufOOB;
    const int k = (wave * 4 + p) * 4 + (lane >> 4);
    const int bc = 8 * ((lane & 15) ^ b_mask(k));
    b_off[p] = (uint32_t)((k * ldb + bc) * 2);
    if (kRagged && n0 + bc >= N) b_off[p] = kBufOOB;
  }
  const char* a_tile = reinterpret_cast<const char*>(A + (long long)m0 * lda);
  const char* b_tile = reinterpret_cast<const char*>(B + n0);
  const long long b_step = (long long)kBK * ldb * 2;
  const uint32_t lds0 = lds_addr(lds);
  constexpr uint32_t kStage = 2 * kOperand;
  auto issue_piece = [&](int kt, int stage, int piece) __attribute__((always_inline)) {
    const uint32_t dst = lds0 + stage * kStage + wave * 4096;
    if (piece < 4) {
      const char* src = a_tile + (long long)kt * kBK * 2;
      if constexpr (kRagged) buf2lds16_s(kt * kBK + a_k[piece & 1] < K ? a_off[piece] : kBufOOB, src, dst + piece * 1024);
      else g2lds16_s(a_off[piece], src, dst + piece * 1024);
    } else {
      const int p = piece - 4;
      const char* src = b_tile + kt * b_step;
      if constexpr (kRagged)
        buf2lds16_s(kt * kBK + (wave * 4 + p) * 4 + (lane >> 4) < K ? b_off[p] : kBufOOB, src, dst + kOperand + p * 1024);
      else g2lds16_s(b_off[p], src, dst + kOperand + p * 1024);
    }
  };

  // ---- fragments of step ks: lhs block i = rows wm*64 + 16 i + lane%16, chunk 4 ks + lane/16;
  // rhs block j = columns wn*64 + 16 j + lane%16, k-rows 32 ks + 8 (lane/16) + 0..7 ----
  const int l16 = lane & 15, lg = lane >> 4;
  uint32_t a_rd[2], b_rd[4];
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) a_rd[ks] = lds0 + (wm * 64 + l16) * 128 + 16 * ((4 * ks + lg) ^ a_swz(l16));
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int n = wn * 64 + j * 16 + 4 * (l16 & 3);
    const int k = 8 * lg + (l16 >> 2);
    b_rd[j] = lds0 + kOperand + k * 256 + (((n >> 3) ^ b_mask(k)) * 16) + (n & 7) * 2;
  }
  struct Frags {
    u32x4 a[4], b[4];
  };
  auto read_step = [&](int stage, int ks, Frags& f, int r) __attribute__((always_inline)) {  // rhs first
    if (r < 4) {
      // k-rows + 4: the same mask; + 32 (ks): the same mask
      const uint32_t ad = b_rd[r] + stage * kStage + ks * 32 * 256;
      const s16x4 v0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(uintptr_t)ad);
      const s16x4 v1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
          (__attribute__((address_space(3))) s16x4*)(uintptr_t)(ad + 4 * 256));
      const u32x2 w0 = __builtin_bit_cast(u32x2, v0), w1 = __builtin_bit_cast(u32x2, v1);
      f.b[r] = u32x4{w0[0], w0[1], w1[0], w1[1]};
    } else {
      f.a[r - 4] = *(const __attribute__((address_space(3))) u32x4*)(uintptr_t)(a_rd[ks] + stage * kStage + (r - 4) * 2048);
    }
  };

  f32x4 acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  const int nk = (K + kBK - 1) / kBK;
#pragma unroll
  for (int st = 0; st < kStages; ++st)
    if (st < nk)
#pragma unroll
      for (int p = 0; p < kPieces; ++p) issue_piece(st, st, p);
  {
    const int younger = min(kStages, nk) - 1;
    if (younger >= 3) wait_and_barrier<3 * kPieces>();
    else if (younger == 2) wait_and_barrier<2 * kPieces>();
    else if (younger == 1) wait_and_barrier<kPieces>();
    else wait_and_barrier<0>();
  }
  Frags fr[2];  // step ks of every slice uses fr[ks]
#pragma unroll
  for (int r = 0; r < 8; ++r) read_step(0, 0, fr[0], r);

  // Slice kt in stage S. kSteady: slices up to kt + kStages exist. Its refill (slice kt +
  // kStages) takes its own stage after the barrier: pieces 0-3 in step 1, 4-7 in the next
  // slice's step 0.
  auto slice = [&](int kt, auto stage_tag, auto steady_tag) __attribute__((always_inline)) {
    constexpr int S = decltype(stage_tag)::value;
    constexpr bool kSteady = decltype(steady_tag)::value != 0;
    constexpr int kPrev = (S + kStages - 1) % kStages, kNext = (S + 1) % kStages;
    const bool more = kSteady || kt + 1 < nk;
    const bool refill0 = kSteady ? true : kt >= 1 && kt - 1 + kStages < nk;
    const bool refill1 = kSteady || kt + kStages < nk;
    static_for<16>([&](auto idx_tag) __attribute__((always_inline)) {
      constexpr int idx = decltype(idx_tag)::value;
      acc[idx >> 2][idx & 3] = H::mfma16(fr[0].b[idx & 3], fr[0].a[idx >> 2], acc[idx >> 2][idx & 3]);
      if constexpr (idx < 8) read_step(S, 1, fr[1], idx);
      if constexpr (idx % 4 == 3)
        if (refill0) issue_piece(kt - 1 + kStages, kPrev, 4 + idx / 4);
      __builtin_amdgcn_sched_barrier(0);
    });
    if (more) {
      // slice kt + 1 has landed: at most slices kt + 2 .. kt + kStages - 1 in flight
      if constexpr (kSteady) {
        wait_and_barrier<(kStages - 2) * kPieces>();
      } else {
        const int younger = min(kStages - 2, nk - 2 - kt);
        if (younger >= 2) wait_and_barrier<2 * kPieces>();
        else if (younger == 1) wait_and_barrier<kPieces>();
        else wait_and_barrier<0>();
      }
    }
    static_for<16>([&](auto idx_tag) __attribute__((always_inline)) {
      constexpr int idx = decltype(idx_tag)::value;
      acc[idx >> 2][idx & 3] = H::mfma16(fr[1].b[idx & 3], fr[1].a[idx >> 2], acc[idx >> 2][idx & 3]);
      if constexpr (idx < 8)
        if (more) read_step(kNext, 0, fr[0], idx);
      if constexpr (idx % 4 == 3)
        if (refill1) issue_piece(kt + kStages, S, idx / 4);
      __builtin_amdgcn_sched_barrier(0);
    });
  };
  auto turn = [&](int kt0, auto steady_tag) __attribute__((always_inline)) {
    static_for<kStages>([&](auto u_tag) __attribute__((always_inline)) {
      constexpr int u = decltype(u_tag)::value;
      if (decltype(steady_tag)::value == 1 || kt0 + u < nk) slice(kt0 + u, gemmp::StageIdx<u>{}, steady_tag);
    });
  };
  // the first turn has no refill in its first slice's step 0 (the prologue filled every stage)
  int kt = 0;
  if (nk > 0) {
    turn(0, Int<0>{});
    kt = kStages;
  }
  for (; kt + 2 * kStages <= nk; kt += kStages) turn(kt, Int<1>{});
  for (; kt < nk; kt += kStages) turn(kt, Int<0>{});

  // ---- epilogue: lane holds C[m = l16][n = 4 lg .. +3] of each block. Each wave packs its quarter
  // (bias added, rounded once) into an LDS region of its own, 64 rows of 128 bytes, chunk c of
  // row r at c ^ (r % 8), and writes whole row segments, 16 bytes per lane ----
  wait_and_barrier<0>();
  const uint32_t region = lds0 + wave * 8192;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int n = n0 + wn * 64 + j * 16 + 4 * lg;
    float bv[4] = {0.f, 0.f, 0.f, 0.f};
    if constexpr (kBias != 0) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int nb = kRagged ? min(n + e, N - 1) : n + e;
        bv[e] = kBias == 1 ? static_cast<const float*>(bias)[nb] : H::to_float(static_cast<const uint16_t*>(bias)[nb]);
      }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      u32x2 packed;
      packed[0] = H::pack2(acc[i][j][0] + bv[0], acc[i][j][1] + bv[1]);
      packed[1] = H::pack2(acc[i][j][2] + bv[2], acc[i][j][3] + bv[3]);
      const int r = 16 * i + l16;
      const uint32_t ad = region + r * 128 + (((2 * j + (lg >> 1)) ^ (r & 7)) * 16) + (lg & 1) * 8;
      *(__attribute__((address_space(3))) u32x2*)(uintptr_t)ad = packed;
    }
  }
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    const int r = 8 * q + (lane >> 3);
    const int c = lane & 7;
    const u32x4 v = *(const __attribute__((address_space(3))) u32x4*)(uintptr_t)(region + r * 128 + ((c ^ (r & 7)) * 16));
    const int m = m0 + wm * 64 + r, n = n0 + wn * 64 + 8 * c;
    if (kRagged && (m >= M || n >= N)) continue;
    __builtin_nontemporal_store(v, reinterpret_cast<u32x4*>(C + (long long)m * ldc + n));
  }
}

// bias_kind: 0 none, 1 fp32, 2 16-bit.
template <typename Tag, int kStages, bool kRagged>
hipError_t launch_gemm_mid(const uint16_t* A, const uint16_t* B, uint16_t* C, const void* bias, int bias_kind, int M,
                           int N, int K, long long lda, long long ldb, long long ldc, hipStream_t stream) {
  const int grid = ((M + gemmm::kT - 1) / gemmm::kT) * ((N + gemmm::kT - 1) / gemmm::kT);
#define KG_GEMM_MID(BIAS)                                                                                       \
  hipLaunchKernelGGL((gemm_mid_kernel<Tag, BIAS, kStages, kRagged>), dim3(grid), dim3(gemmm::kThreads), 0, stream, A, B, \
                     C, bias, M, N, K, lda, ldb, ldc)
  if (bias_kind == 0) KG_GEMM_MID(0);
  else if (bias_kind == 1) KG_GEMM_MID(1);
  else KG_GEMM_MID(2);
#undef KG_GEMM_MID
  return hipGetLastError();
}

}  // namespace kg_gfx950
