// Implicit-GEMM conv2d on gfx950 matrix cores over a channel-last copy of the image, for any
// NCHW shape, kernel size, stride, dilation and padding: bf16/f16 (v_mfma_f32_16x16x32) or
// fp32 (v_mfma_f32_16x16x4_f32) operands, fp32 accumulation. Two launches:
//
// conv_pack_kernel writes, into the stream's workspace, the part of the zero-padded images
// that the windows touch as [n][row][column][channel] (channels rounded up with zeros to
// 16 bytes) and the weights as [filter][(kh, kw, c)], rows rounded up with zeros to 128 bytes.
//
// conv2d_nhwc_kernel is then a GEMM of output pixels x filters in which both operands are
// k-contiguous: 16 bytes of one tap's channels are one chunk, a pixel's chunk k lies at the
// pixel's window origin plus an offset that depends on k only, and nothing has to be tested
// against the image's edges. So both operands go HBM/L2 -> LDS by buffer_load ... lds (no
// registers, no per-element gather: the gather of conv2d_igemm_kernel, one 2-byte load and its
// bounds test per element, kept its matrix cores idle over 95 % of the time on rows that are
// no whole 4-pixel pieces).
#pragma once

#include <type_traits>

#include "common.h"
#include "conv2d.h"
#include "conv2d_igemm.h"
#include "lds_dma.h"

namespace kg_gfx950 {

namespace convn {
constexpr int kThreads = 256;  // 4 waves, 2 x 2
constexpr int kRowBytes = 128;  // K slice: 8 chunks of 16 bytes per row

struct Geometry {
  int n, c, h, w, f, kh, kw, pt, pl;  // the conv (n: images of this launch)
  int cp;         // channels per pixel of the copy
  int hp, wp;     // its rows and columns per image
  int col_up;     // pieces of the copy's rows start at columns -col_up + V i of the image
  int row_step;   // image rows per row of the copy (one kernel row: only the rows it meets)
  int paired;     // 16-bit, cp = 4: one chunk is two neighbouring pixels
  int taps_w;     // runs per kernel row: 1 (a run is the row, dilation_w 1) or KW (a run is a tap)
  int cpr;        // 16-byte chunks of a run
  int halves;     // runs of at most 4 chunks: a slice is two halves, of 4 chunks each
  int spr, hpr;   // slices (or halves) of a run, the last one padded
  int slices;     // K slices
  int P, NP;      // Ho Wo, n Ho Wo
  uint32_t off_kh, off_kw;      // bytes between kernel rows, taps
  uint32_t row_h, row_w, img;   // bytes between output rows, output pixels, images
  uint32_t x_bytes;             // the copy's size
  uint32_t w_pitch;             // bytes per packed filter row
  int bias_kind;  // 0 none, 1 fp32, 2 same dtype; +2: one value per pixel instead of per filter
  int kcs;        // split-K: slices per split; 0 = all of them
  int out_pitch;  // elements between filter rows of an image's output (Ho Wo)
  int piece;      // output pixels per store: 8, 4 or 1 (rows start and end on multiples of it)
  FastDiv div_p, div_wo, div_spr, div_hpr, div_taps_w, div_pieces, div_hp, div_cpx, div_wrow, div_cp;
};

// LDS rows are 128 bytes, two per 256-byte bank line: the 16 rows of a fragment read take 16
// distinct slots when chunk c of row r sits at c ^ ((r >> 1) & 7).
__device__ __forceinline__ int swz(int row) { return (row >> 1) & 7; }
// n / d for n < 2^31 (fdiv's sum then stays below 2^32)
__device__ __forceinline__ uint32_t fdiv31(uint32_t n, FastDiv f) { return (__umulhi(n, f.mul) + n) >> f.shift; }
}  // namespace convn

// 16 bytes from an address of any element alignment.
__device__ __forceinline__ u32x4 ld16_any(const void* p) {
  u32x4 v;
  __builtin_memcpy(&v, p, 16);
  return v;
}

// Blocks below x_blocks: a thread copies a block of V channels x V neighbouring pixels of one
// image row (V = 8, fp32 4): V row pieces of 16 bytes in, transposed in registers, V pixels'
// chunks of 16 bytes out, the channel blocks of a pixel piece in neighbouring threads. Pixels of
// the padding are zeros; a piece that crosses a row's end reads on into the next row and
// its pixels there are not used, and only a piece that crosses the tensor's ends is read by
// elements. (With 2-byte loads per element, 15x408x85x85 took 100 us, 1.7 TB/s.)
// Paired pixels: a thread reads two pixels by elements and writes their one chunk (whole rows of
// chunks per wave; 8 pixels per thread wrote 8 pieces 64 bytes apart: 14 against 10 us for
// 32x3x224x224).
// Other blocks: one 16-byte chunk of the packed weights per thread.
template <typename Tag>
__global__ __launch_bounds__(convn::kThreads) void conv_pack_kernel(
    const typename convg::IgElem<Tag>::T* __restrict__ x, const typename convg::IgElem<Tag>::T* __restrict__ wt,
    u32x4* __restrict__ xp, u32x4* __restrict__ wp, convn::Geometry s, int x_blocks) {
  using E = convg::IgElem<Tag>;
  using T = typename E::T;
  constexpr int V = E::kPerChunk;
  if (V == 8 && s.paired && (int)blockIdx.x < x_blocks) {
    const uint32_t idx = blockIdx.x * convn::kThreads + threadIdx.x;
    const uint32_t row = fdiv(idx, s.div_pieces);  // pairs of a row
    const int wi = (int)(idx - row * s.div_pieces.d) * 2 - s.pl;
    const uint32_t n = fdiv(row, s.div_hp);
    if ((int)n >= s.n) return;
    const int hi = (int)(row - n * s.hp) * s.row_step - s.pt;
    const long long hw = (long long)s.h * s.w;
    const T* src = x + (long long)n * s.c * hw + (long long)hi * s.w + wi;
    T v[V];
#pragma unroll
    for (int e = 0; e < V; ++e) {
      const int c = e & 3, u = e >> 2;
      const bool ok = (unsigned)hi < (unsigned)s.h && (unsigned)(wi + u) < (unsigned)s.w && c < s.c;
      v[e] = ok ? src[c * hw + u] : T(0);
    }
    u32x4 out;
    __builtin_memcpy(&out, v, 16);
    xp[idx] = out;
    return;
  }
  if ((int)blockIdx.x < x_blocks) {
    const uint32_t idx = blockIdx.x * convn::kThreads + threadIdx.x;
    const uint32_t piece = fdiv(idx, s.div_cpx);
    const uint32_t cb = idx - piece * s.div_cpx.d;  // channel block
    const uint32_t row = fdiv(piece, s.div_pieces);  // n hp + row of the copy
    const int wi = (int)(piece - row * s.div_pieces.d) * V - s.col_up;  // the piece's first column
    const int col0 = wi + s.pl;                                          // and in the copy
    const uint32_t n = fdiv(row, s.div_hp);
    if ((int)n >= s.n) return;
    const int hi = (int)(row - n * s.hp) * s.row_step - s.pt;
    const long long hw = (long long)s.h * s.w;  // (a plane may have 2^31 elements: only the copy is bounded)
    const int c0 = (int)cb * V;
    u32x4 in[V], out[V];
#pragma unroll
    for (int e = 0; e < V; ++e) in[e] = u32x4{0, 0, 0, 0};
    if ((unsigned)hi < (unsigned)s.h && wi < s.w && wi + V > 0) {
      const long long first = ((long long)n * s.c + c0) * hw + (long long)hi * s.w + wi;  // element of x
      const long long last = (long long)s.n * s.c * hw - V;
#pragma unroll
      for (int e = 0; e < V; ++e) {
        const long long at = first + e * hw;
        if (c0 + e < s.c) {
          if (at >= 0 && at <= last) {
            in[e] = ld16_any(x + at);
          } else {
            T v[V];
#pragma unroll
            for (int u = 0; u < V; ++u) v[u] = (unsigned)(wi + u) < (unsigned)s.w ? x[at + u] : T(0);
            __builtin_memcpy(&in[e], v, 16);
          }
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
      if ((unsigned)(wi + u) >= (unsigned)s.w) out[u] = u32x4{0, 0, 0, 0};
    u32x4* dst = xp + ((long long)row * s.wp + col0) * (int)s.div_cpx.d + cb;
#pragma unroll
    for (int u = 0; u < V; ++u)
      if ((unsigned)(col0 + u) < (unsigned)s.wp) dst[u * (int)s.div_cpx.d] = out[u];
    return;
  }
  const uint32_t idx = (blockIdx.x - x_blocks) * convn::kThreads + threadIdx.x;
  const uint32_t f = fdiv(idx, s.div_wrow);
  if ((int)f >= s.f) return;
  const uint32_t q = idx - f * s.div_wrow.d;
  const uint32_t run = s.halves ? fdiv(q >> 2, s.div_hpr) : fdiv(q >> 3, s.div_spr);
  const uint32_t chunk = s.halves ? q - run * s.hpr * 4 : q - run * s.spr * 8;  // of the run
  const uint32_t kh = fdiv(run, s.div_taps_w);
  const int kw0 = (int)(run - kh * s.taps_w);  // the run's first tap column
  const int taps = s.taps_w == 1 ? s.kw : 1;
  T v[V];
#pragma unroll
  for (int e = 0; e < V; ++e) v[e] = T(0);
  if ((int)kh < s.kh && (int)chunk < s.cpr) {
#pragma unroll
    for (int e = 0; e < V; ++e) {
      const uint32_t tap = fdiv(chunk * V + e, s.div_cp);
      const int c = (int)(chunk * V + e - tap * s.cp);
      if (c < s.c && (int)tap < taps) v[e] = wt[(((long long)f * s.c + c) * s.kh + kh) * s.kw + kw0 + (int)tap];
    }
  }
  u32x4 out;
  __builtin_memcpy(&out, v, 16);
  wp[idx] = out;
}

// Tiles of BM pixels x BN filters, 4 waves of BM/2 x BN/2; 16 x 16 blocks; K slices of 8 chunks
// through an LDS ring of kRing stages. A slice is 64 or 128 MFMA cycles of work for a wave, so
// its other instructions count: the taps' offsets are wave-uniform (one scalar per slice; a
// per-lane offset and its divisions made a slice 190 instructions and 1000 cycles of issue),
// and several small workgroups share a CU, one's MFMAs under another's waits.
// kHalves: runs of at most 4 chunks; a slice is two runs' halves and the lanes of its two halves
// take an offset each.
// Split-K (s.kcs > 0): workgroup row y runs slices [y kcs, (y+1) kcs) and stores fp32 sums
// without bias to partial[y][n][f][Ho Wo] (added in y order by conv_splitk_reduce_kernel).
template <typename Tag, int BM, int BN, int kRing, bool kHalves>
__global__ __launch_bounds__(convn::kThreads, 2) void conv2d_nhwc_kernel(
    const char* __restrict__ xp, const char* __restrict__ wp, typename convg::IgElem<Tag>::T* __restrict__ y,
    const void* __restrict__ bias, convn::Geometry s, float* __restrict__ partial) {
  using namespace convn;
  using E = convg::IgElem<Tag>;
  using T = typename E::T;
  constexpr int V = E::kPerChunk;
  constexpr int MA = BM / 32, NB = BN / 32;       // 16-row blocks per wave
  constexpr int kStage = (BM + BN) * kRowBytes;
  constexpr int PA = BM / 32, PB = BN / 32;       // copies per wave and slice (8 rows each)
  static_assert(BN * BM * 2 <= kRing * kStage, "a tile's 16-bit outputs fit in the ring");
  __shared__ __attribute__((aligned(1024))) char lds[kRing * kStage];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  // each XCD takes one contiguous range of tiles: the filter tiles of one pixel tile are
  // adjacent, and neighbouring pixel tiles share rows of the copy in its L2
  const int tiles_f = (s.f + BN - 1) / BN;
  const int total = gridDim.x;
  const int xcd = blockIdx.x % 8;
  const int logical = xcd * (total / 8) + min(xcd, total % 8) + blockIdx.x / 8;
  const int f0 = (logical % tiles_f) * BN;
  const int j0 = (logical / tiles_f) * BM;
  int kt0 = 0, nk = s.slices;
  if (s.kcs > 0) {
    kt0 = blockIdx.y * s.kcs;
    nk = min(nk - kt0, s.kcs);
    partial += (long long)blockIdx.y * s.NP * s.f;
  }

  // ---- HBM -> LDS copies: copy p of a wave covers rows (wave*P + p)*8 + lane/8 of its
  // operand, LDS slot lane%8, which holds chunk slot ^ swz(row). Rows 8 apart differ in bit 2
  // of swz: a lane's copies hold chunk c_even (even copies) or c_even ^ 4 ----
  static_assert(PA % 2 == 0 && PB % 2 == 0, "a wave's first copy row is a multiple of 16");
  const int slot = lane & 7;
  const int c_even = slot ^ swz(lane >> 3);
  uint32_t a_off[PA], b_off[PB];
#pragma unroll
  for (int p = 0; p < PA; ++p) {
    const int row = (wave * PA + p) * 8 + (lane >> 3);
    const uint32_t j = (uint32_t)min(j0 + row, s.NP - 1);
    const uint32_t n = fdiv(j, s.div_p);
    const uint32_t pix = j - n * s.P;
    const uint32_t ho = fdiv(pix, s.div_wo);
    const int c = c_even ^ (4 * (p & 1));
    a_off[p] = n * s.img + ho * s.row_h + (pix - ho * s.div_wo.d) * s.row_w + 16 * (kHalves ? c & 3 : c);
  }
#pragma unroll
  for (int p = 0; p < PB; ++p) {
    const int row = (wave * PB + p) * 8 + (lane >> 3);
    b_off[p] = (uint32_t)min(f0 + row, s.f - 1) * s.w_pitch + 16 * (c_even ^ (4 * (p & 1)));
  }
  const uint32_t lds0 = lds_addr(lds);
  const uint32_t a_dst = lds0 + wave * PA * 1024, b_dst = lds0 + BM * kRowBytes + wave * PB * 1024;

  // The place in the contraction of the next copies: unit `at` (a slice of 8 chunks, kHalves:
  // a half of 4) of the run that starts `off` bytes from every window's origin.
  const int units = kHalves ? s.hpr : s.spr;  // per run
  uint32_t off;
  int at, kw, kh, kt = kt0;
  {
    const uint32_t u = kHalves ? 2 * kt0 : kt0;
    const uint32_t run = fdiv31(u, kHalves ? s.div_hpr : s.div_spr);
    kh = (int)fdiv31(run, s.div_taps_w);
    kw = (int)run - kh * s.taps_w;
    at = (int)u - (int)run * units;
    off = (uint32_t)kh * s.off_kh + (uint32_t)kw * s.off_kw + (uint32_t)at * (kHalves ? 64 : 128);
  }
  const uint32_t to_next_kw = s.off_kw - (uint32_t)units * (kHalves ? 64 : 128);
  const uint32_t to_next_kh = s.off_kh - (uint32_t)s.taps_w * s.off_kw;
  auto advance = [&]() __attribute__((always_inline)) {
    off += kHalves ? 64 : 128;
    if (++at == units) {
      at = 0;
      off += to_next_kw;
      if (++kw == s.taps_w) {
        kw = 0;
        ++kh;
        off += to_next_kh;
      }
    }
  };
  // A chunk past its run's end (kHalves: or past the last run) is not read: its offset lies
  // outside the buffer and zeros land in LDS (its weights are zeros too, but the bytes there may
  // be infinities). An origin plus kBufOOB stays outside: the copy is smaller than 2^31 bytes.
  uint32_t k_off[2];  // of the even and the odd copies
  auto slice_offsets = [&]() __attribute__((always_inline)) {
    if constexpr (kHalves) {
      uint32_t o[2];
      int valid[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        o[i] = off;
        valid[i] = kh < s.kh ? s.cpr - 4 * at : 0;
        advance();
      }
      const bool hi = (c_even & 4) != 0;
      const int c3 = c_even & 3;
      k_off[0] = c3 < (hi ? valid[1] : valid[0]) ? (hi ? o[1] : o[0]) : kBufOOB;
      k_off[1] = c3 < (hi ? valid[0] : valid[1]) ? (hi ? o[0] : o[1]) : kBufOOB;
    } else {
      const int valid = s.cpr - 8 * at;
      k_off[0] = k_off[1] = off;
      if (valid < 8) {
        k_off[0] = c_even < valid ? off : kBufOOB;
        k_off[1] = (c_even ^ 4) < valid ? off : kBufOOB;
      }
      advance();
    }
    ++kt;
  };
  auto issue_piece = [&](uint32_t stage_bytes, int p) __attribute__((always_inline)) {
    if (p < PA)
      buf2lds16_r(a_off[p] + k_off[p & 1], xp, s.x_bytes, a_dst + stage_bytes + p * 1024);
    else
      g2lds16_s(b_off[p - PA], wp + (kt - 1) * kRowBytes, b_dst + stage_bytes + (p - PA) * 1024);
  };

  // ---- fragments: lane l holds 16 bytes (chunk 4 ks + l/16) of row l%16 of a block ----
  const int l16 = lane & 15, lg = lane >> 4;
  uint32_t a_rd[2], b_rd[2];
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) {  // blocks are 16 rows apart: the same swz
    const int c = (4 * ks + lg) ^ swz(l16);
    a_rd[ks] = lds0 + (wm * (BM / 2) + l16) * kRowBytes + 16 * c;
    b_rd[ks] = lds0 + BM * kRowBytes + (wn * (BN / 2) + l16) * kRowBytes + 16 * c;
  }
  auto lds_read = [&](uint32_t at_byte) -> u32x4 {
    return *(const __attribute__((address_space(3))) u32x4*)(uintptr_t)at_byte;
  };

  // fp32: one set of accumulators per element of the chunk, added at the end: sums a quarter
  // as long (the rounding of a 2304-term sum: 4.2e-7 of the result against 8.3e-7 in one)
  constexpr int KA = V == 4 ? 4 : 1;
  f32x4 acc[KA][MA][NB];
#pragma unroll
  for (int e = 0; e < KA; ++e)
#pragma unroll
    for (int i = 0; i < MA; ++i)
#pragma unroll
      for (int j = 0; j < NB; ++j) acc[e][i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

#pragma unroll
  for (int st = 0; st < kRing - 1; ++st)
    if (st < nk) {
      slice_offsets();
#pragma unroll
      for (int p = 0; p < PA + PB; ++p) issue_piece(st * kStage, p);
    }

  constexpr int kSteps = 2 * MA * NB;          // 16 x 16 blocks x k steps of a slice
  constexpr int kReads = MA + NB;              // fragments of a k step
  constexpr int kGap = kSteps / (PA + PB);     // steps between copies
  static_assert(kGap >= 1, "copy slots");
  uint32_t rd = 0, fill = (kRing - 1) * kStage;  // stage read, stage filled
  auto slice = [&](int it, auto refill_tag) __attribute__((always_inline)) {
    constexpr bool kRefill = decltype(refill_tag)::value != 0;
    u32x4 af[2][MA], bf[2][NB];
    const uint32_t ar[2] = {a_rd[0] + rd, a_rd[1] + rd}, br[2] = {b_rd[0] + rd, b_rd[1] + rd};
    auto read = [&](int ks, int r) __attribute__((always_inline)) {  // rhs fragments first
      if (r < NB) bf[ks][r] = lds_read(br[ks] + r * 16 * kRowBytes);
      else af[ks][r - NB] = lds_read(ar[ks] + (r - NB) * 16 * kRowBytes);
    };
    if constexpr (kRefill) slice_offsets();
#pragma unroll
    for (int r = 0; r < kReads; ++r) read(0, r);
    __builtin_amdgcn_sched_barrier(0);
    // the blocks' MFMAs, with the second k step's fragment reads and the refill copies
    // slotted between them (a burst of copies stalls its wave 60-100 cycles each)
    static_for<kSteps>([&](auto idx_tag) __attribute__((always_inline)) {
      constexpr int idx = decltype(idx_tag)::value;
      constexpr int ks = idx / (MA * NB), i = idx % (MA * NB) / NB, j = idx % NB;
      if constexpr (V == 8 && idx % (MA * NB) == 0) {
        // paired pixels: an odd kernel row ends in the middle of a chunk, and the pixel after it
        // (any value, infinities included) must not meet the weights' zeros
        if (s.paired && (s.kw & 1)) {
          const uint32_t u = kHalves ? 2 * (kt0 + it) + ks : kt0 + it;  // this step's half, this slice
          const int in_run = (int)(u - fdiv31(u, kHalves ? s.div_hpr : s.div_spr) * units);
          const uint32_t keep = (kHalves ? 4 * in_run : 8 * in_run + 4 * ks) + lg == s.cpr - 1 ? 0u : ~0u;
#pragma unroll
          for (int b = 0; b < MA; ++b) {
            af[ks][b][2] &= keep;
            af[ks][b][3] &= keep;
          }
        }
      }
      if constexpr (V == 8) {
        acc[0][i][j] = Half16<Tag>::mfma16(af[ks][i], bf[ks][j], acc[0][i][j]);
      } else {
        // one k per lane: MFMA e takes element e of each lane's chunk, in both operands
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const uint32_t au = af[ks][i][e], bu = bf[ks][j][e];
          acc[e][i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(__builtin_bit_cast(float, au),
                                                              __builtin_bit_cast(float, bu), acc[e][i][j], 0, 0, 0);
        }
      }
      if constexpr (idx < MA * NB) {  // the reads of step 1 spread over step 0
        constexpr int lo = kReads * idx / (MA * NB), hi = kReads * (idx + 1) / (MA * NB);
#pragma unroll
        for (int r = lo; r < hi; ++r) read(1, r);
      }
      if constexpr (kRefill && idx % kGap == kGap - 1 && idx / kGap < PA + PB) issue_piece(fill, idx / kGap);
      __builtin_amdgcn_sched_barrier(0);
    });
    rd = rd == (kRing - 1) * kStage ? 0 : rd + kStage;
    if constexpr (kRefill) fill = fill == (kRing - 1) * kStage ? 0 : fill + kStage;
  };
  int it = 0;
  for (; it + kRing - 1 < nk; ++it) {
    // slice it has landed (the younger ones may be in flight) and every wave is done with the
    // slice before it, whose stage takes the next copies
    wait_and_barrier<(kRing - 2) * (PA + PB)>();
    slice(it, Int<1>{});
  }
  for (; it < nk; ++it) {
    wait_and_barrier<0>();
    slice(it, Int<0>{});
  }

  // ---- epilogue: lane holds pixels 4 lg .. +3 of filter l16 of each block. 16-bit outputs go
  // through LDS (the ring) as [filter][pixel] so that Y is written in whole row pieces; 16-byte
  // chunk c of filter row f at c ^ out_mask(f) ----
  const bool split = s.kcs > 0;
  auto out_mask = [](int f) { return BM == 128 ? f & 15 : (f >> 1) & 7; };
  if (V == 8 && !split) __syncthreads();
#pragma unroll
  for (int j = 0; j < NB; ++j) {
    const int fr = wn * (BN / 2) + 16 * j + l16;
    const int f = f0 + fr;
    auto bias_at = [&](int b) {
      return s.bias_kind & 1 ? static_cast<const float*>(bias)[b] : E::to_float(static_cast<const T*>(bias)[b]);
    };
    const float bv = !split && (s.bias_kind == 1 || s.bias_kind == 2) ? bias_at(min(f, s.f - 1)) : 0.f;
#pragma unroll
    for (int i = 0; i < MA; ++i) {
      const int px = wm * (BM / 2) + 16 * i + 4 * lg;
      f32x4 r = acc[0][i][j];
      if constexpr (KA == 4) r = (acc[0][i][j] + acc[1][i][j]) + (acc[2][i][j] + acc[3][i][j]);
#pragma unroll
      for (int e = 0; e < 4; ++e) r[e] += bv;
      if (!split && s.bias_kind > 2) {
#pragma unroll
        for (int e = 0; e < 4; ++e) r[e] += bias_at(min(j0 + px + e, s.NP - 1));
      }
      if (V == 4 || split) {
        // fp32 outputs or partial sums: straight from the registers
        float* out = split ? partial : reinterpret_cast<float*>(y);
        const long long pitch = split ? s.P : s.out_pitch;
        if (f < s.f) {
          if (split ? (s.P & 3) == 0 : s.piece >= 4) {
            const int jv = j0 + px;
            if (jv < s.NP) {
              const uint32_t n = fdiv((uint32_t)jv, s.div_p);
              *reinterpret_cast<f32x4*>(out + ((long long)n * s.f + f) * pitch + (jv - n * s.P)) = r;
            }
          } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const int jv = j0 + px + e;
              if (jv < s.NP) {
                const uint32_t n = fdiv((uint32_t)jv, s.div_p);
                out[((long long)n * s.f + f) * pitch + (jv - n * s.P)] = r[e];
              }
            }
          }
        }
      } else {
        using P2 = Half16<typename std::conditional<V == 8, Tag, Bf16Tag>::type>;
        u32x2 packed;
        packed[0] = P2::pack2(r[0], r[1]);
        packed[1] = P2::pack2(r[2], r[3]);
        *reinterpret_cast<u32x2*>(lds + fr * (BM * 2) + ((px >> 3) ^ out_mask(fr)) * 16 + (px & 4) * 2) = packed;
      }
    }
  }
  if (V == 8 && !split) {
    __syncthreads();
    // rows of BM pixels, G per lane
    auto store_rows = [&](auto g_tag) {
      constexpr int G = decltype(g_tag)::value;
      using Piece = typename std::conditional<G == 8, u32x4, typename std::conditional<G == 4, u32x2, uint16_t>::type>::type;
      constexpr int kLanes = BM / G;             // threads per row
      constexpr int kRows = kThreads / kLanes;   // rows per pass
      const int px = (tid % kLanes) * G;
      const int j = j0 + px;
      if (j >= s.NP) return;
      const uint32_t n = fdiv((uint32_t)j, s.div_p);
      const uint32_t p = j - n * s.P;
      uint16_t* out = reinterpret_cast<uint16_t*>(y) + (long long)n * s.f * s.out_pitch + p;
#pragma unroll 4
      for (int r = tid / kLanes; r < BN; r += kRows) {
        if (f0 + r >= s.f) break;
        *reinterpret_cast<Piece*>(out + (long long)(f0 + r) * s.out_pitch) =
            *reinterpret_cast<const Piece*>(lds + r * (BM * 2) + ((px >> 3) ^ out_mask(r)) * 16 + (px & 7) * 2);
      }
    };
    if (s.piece == 8) store_rows(Int<8>{});
    else if (s.piece == 4) store_rows(Int<4>{});
    else store_rows(Int<1>{});
  }
}

// The copy's layout for `images` images of conv s (es: bytes per element).
inline convn::Geometry conv_nhwc_geometry(const ConvShape& s, int images, int es) {
  convn::Geometry g;
  const int V = 16 / es;
  g.n = images; g.c = s.c; g.h = s.h; g.w = s.w; g.f = s.f; g.kh = s.kh; g.kw = s.kw; g.pt = s.pt; g.pl = s.pl;
  // up to four 16-bit channels under an even column stride: 4 channels per pixel, so that a
  // window's row (KW pixels) is one run of 8-byte pixels that starts on 16 bytes
  g.paired = es == 2 && s.c <= 4 && s.sw % 2 == 0 && s.dw == 1;
  g.cp = g.paired ? 4 : (s.c + V - 1) / V * V;
  g.row_step = s.kh == 1 ? s.sh : 1;
  g.hp = s.kh == 1 ? s.ho : (s.ho - 1) * s.sh + (s.kh - 1) * s.dh + 1;
  g.wp = (s.wo - 1) * s.sw + (s.kw - 1) * s.dw + 1;
  if (g.paired) g.wp = (g.wp + 2) / 2 * 2;  // the last chunk of a window's row may reach one pixel past it
  g.taps_w = s.dw == 1 ? 1 : s.kw;
  g.cpr = ((s.dw == 1 ? s.kw : 1) * g.cp + V - 1) / V;
  g.halves = g.cpr <= 4;
  g.hpr = (g.cpr + 3) / 4;
  g.spr = (g.cpr + 7) / 8;
  g.slices = g.halves ? (s.kh * g.taps_w * g.hpr + 1) / 2 : s.kh * g.taps_w * g.spr;
  g.P = s.ho * s.wo;
  g.NP = images * g.P;
  g.out_pitch = g.P;
  g.piece = g.P % 8 == 0 ? 8 : g.P % 4 == 0 ? 4 : 1;
  const uint32_t px = (uint32_t)(g.cp * es);
  const uint32_t row = (uint32_t)g.wp * px;
  g.off_kh = (uint32_t)s.dh * row;
  g.off_kw = (uint32_t)s.dw * px;
  g.row_h = s.kh == 1 ? row : (uint32_t)s.sh * row;
  g.row_w = (uint32_t)s.sw * px;
  g.img = (uint32_t)g.hp * row;
  g.x_bytes = (uint32_t)images * g.img;
  g.w_pitch = (uint32_t)g.slices * convn::kRowBytes;
  g.bias_kind = 0;
  g.kcs = 0;
  g.div_p = make_fast_div((uint32_t)g.P);
  g.div_wo = make_fast_div((uint32_t)s.wo);
  g.div_spr = make_fast_div((uint32_t)g.spr);
  g.div_hpr = make_fast_div((uint32_t)g.hpr);
  g.div_cp = make_fast_div((uint32_t)g.cp);
  g.div_taps_w = make_fast_div((uint32_t)g.taps_w);
  // pieces at multiples of V columns, aligned to 4 bytes at least, where rows are of even length
  g.col_up = g.paired ? s.pl : s.w % 2 == 0 ? (s.pl + V - 1) / V * V : s.pl;
  const uint32_t px_per = g.paired ? 2 : (uint32_t)V;
  g.div_pieces = make_fast_div(((uint32_t)(g.wp - s.pl + g.col_up) + px_per - 1) / px_per);
  g.div_hp = make_fast_div((uint32_t)g.hp);
  g.div_cpx = make_fast_div(g.paired ? 1u : (uint32_t)(g.cp / V));
  g.div_wrow = make_fast_div(g.w_pitch / 16);
  return g;
}

// How a conv runs on this kernel: images per pass (their copy and the packed weights fit
// max_bytes), tile, split-K. ok = false: not at all. The second launch costs about 3 us and the
// copy moves the image twice, which a small or short contraction's gather does not repay (us,
// this form against the gather):
//   below 4 MFLOP (2x5x13x11, 4 filters: 12.5 / 10.8; 1x16x30x30, 16 filters, 4.1 MFLOP: 12.5 /
//   15.1), fp32, whose MFMAs are slower in both, 100 (15x16x10x10, 192 filters 5x5 s2, 60: 17.7 /
//   15.3; 4x32x14x14, 64 filters 3x3, 29: 12.6 / 15.3; 2x64x50x50 s2, 92: 16 / 16);
//   up to 96 values per output (3x3 of 8 channels: 13-14 / 11-12; of 16: 13.8 / 15.0);
//   under 100 operations per copied value (fp32 9x232x154x154, 16 filters 3x3 s2: 324 / 224);
//   one tap, which reads every pixel once, of few channels or filters or over a copy beyond 48 MiB
//   (1x1 of 408 channels to 16 85 x 85: 76 / 51; of 368 to 64 160 x 37, 65 MB: 53 / 45; of 504 to 128
//   58 x 58 s2, 47 MB: 48 / 56; fp32 of 160 to 128 45 x 57: 59 / 49, of 256 to 128 30 x 30: 25 / 39).
struct ConvNhwcPlan {
  bool ok = false;
  int images = 0;      // per pass
  int bm = 64, ring = 5;  // tiles of bm pixels x 64 filters
  int splits = 1, kcs = 0;
  size_t w_bytes = 0, x_bytes = 0, partial_bytes = 0;
  size_t bytes() const { return w_bytes + x_bytes + partial_bytes; }
};

inline ConvNhwcPlan conv_nhwc_plan(const ConvShape& s, bool f32, long long max_bytes) {
  ConvNhwcPlan p;
  const int es = f32 ? 4 : 2;
  // everything in 64 bits first: the geometry below holds 32-bit byte offsets
  const long long V = 16 / es;
  const long long cp = ((long long)s.c + V - 1) / V * V;
  const long long hp = (long long)(s.ho - 1) * s.sh + (long long)(s.kh - 1) * s.dh + 1;
  const long long wp = (long long)(s.wo - 1) * s.sw + (long long)(s.kw - 1) * s.dw + 3;
  const long long taps = (long long)s.kh * s.kw;
  if (s.ho < 1 || s.wo < 1 || s.n < 1 || s.f < 1 || s.c < 1) return p;
  if (2.0 * s.n * s.f * s.ho * s.wo * s.c * s.kh * s.kw < (f32 ? 1e8 : 4e6)) return p;
  if (taps == 1 ? s.c < (f32 ? 256 : 160) || s.f < (f32 ? 64 : 32) : s.c * taps <= 96) return p;
  if (cp > (1ll << 20) || hp > (1ll << 20) || wp > (1ll << 20) || taps > (1ll << 20)) return p;
  if (cp * es * wp > max_bytes || cp * es * wp * hp > max_bytes) return p;
  const long long w_bytes = (long long)s.f * ((cp * taps * es + 127) / 128 * 128);  // (at least; checked again below)
  if (w_bytes > max_bytes / 2 || (long long)s.ho * s.wo > (1ll << 30)) return p;
  const convn::Geometry g = conv_nhwc_geometry(s, 1, es);
  if (taps == 1 && (long long)s.n * g.img > (48ll << 20)) return p;
  if (2.0 * s.f * g.P * s.c * taps < 100.0 * g.img / es) return p;
  p.w_bytes = (size_t)s.f * g.w_pitch;
  if ((long long)p.w_bytes > max_bytes / 2) return p;
  const long long room = max_bytes - (long long)p.w_bytes;
  long long images = std::min<long long>(s.n, room / (long long)g.img);
  images = std::min(images, ((1ll << 31) - 1) / g.P);
  if (images < 1) return p;
  p.images = (int)images;
  p.x_bytes = (size_t)images * g.img;
  p.ok = true;
  // Tiles of 128 x 64 when they give every CU two workgroups, else 64 x 64 (16-bit N=32 C=256
  // F=256 14 x 14 3x3: 24 us either way; N=8 C=33 F=130 111 x 111 5x5: 71 against 95 us). Two ring stages
  // for contractions of at most 4 slices (7x7 s2 of 3 channels at 224 x 224: 40 against 45 us
  // with three), else three; small grids, one or two workgroups per CU, take five stages,
  // which hide the copies' latency where no other workgroup does (C=512 7 x 7: 34 against 53 us
  // with two).
  const long long np = (long long)images * g.P;
  auto tiles = [&](int bm, int bn) { return ((np + bm - 1) / bm) * ((s.f + bn - 1) / bn); };
  if (tiles(128, 64) >= 512) {
    p.bm = 128;
    p.ring = g.slices <= 4 ? 2 : 3;
  } else {
    p.bm = 64;
    p.ring = tiles(64, 64) > 512 ? 3 : 5;
  }
  // Split-K (whole batches only) by a time model: a slice takes 330 ns (fp32 650) in each round
  // of 512 workgroups, the partials cost 8 bytes per output and split at 2 bytes/ns, the
  // reduction's launch 4 us; chunks of at least 8 slices (fp32 4). N=1 C=512 7 x 7: 29 -> 18 us in 8
  // splits (fp32: 102 -> 29 in 16); N=8 C=256 14 x 14 measures the same split and whole.
  const long long t = tiles(p.bm, 64), nfp = np * s.f, slice_ns = f32 ? 650 : 330;
  if (images == s.n && nfp < (1ll << 31)) {
    long long best = 1, best_ns = (t + 511) / 512 * g.slices * slice_ns;
    for (long long sp = 2; sp <= g.slices / (f32 ? 4 : 8) && t * (sp - 1) < 512; ++sp) {
      const long long ns =
          (t * sp + 511) / 512 * ((g.slices + sp - 1) / sp) * slice_ns + sp * nfp * 8 / 2000 + 4000;
      if (ns < best_ns) { best = sp; best_ns = ns; }
    }
    const int c = (int)((g.slices + best - 1) / best);
    const int splits = (g.slices + c - 1) / c;
    const size_t partial_bytes = (size_t)splits * nfp * 4, x_bytes = (p.x_bytes + 255) / 256 * 256;
    if (splits > 1 && p.w_bytes + x_bytes + partial_bytes <= (size_t)max_bytes) {
      p.kcs = c;
      p.splits = splits;
      p.x_bytes = x_bytes;
      p.partial_bytes = partial_bytes;
    }
  }
  return p;
}

// MFMA instructions of a conv run by `plan` (16-bit: 16x16x32, fp32: 16x16x4).
inline long long conv_nhwc_mfma(const ConvShape& s, const ConvNhwcPlan& plan, bool f32) {
  long long n = 0;
  for (int n0 = 0; n0 < s.n; n0 += plan.images) {
    const convn::Geometry g = conv_nhwc_geometry(s, std::min(plan.images, s.n - n0), f32 ? 4 : 2);
    const long long tiles = (long long)((g.NP + plan.bm - 1) / plan.bm) * ((s.f + 63) / 64);
    n += tiles * g.slices * (plan.bm / 16) * 4 * 2 * (f32 ? 4 : 1);
  }
  return n;
}

// The GEMM launch: tiles of bm pixels x 64 filters on a ring of `ring` stages.
template <typename Tag>
void launch_nhwc_gemm(const char* xp, const char* wp, typename convg::IgElem<Tag>::T* y, const void* bias,
                      const convn::Geometry& g, int bm, int ring, int splits, float* partial, hipStream_t stream) {
  const int grid = ((g.NP + bm - 1) / bm) * ((g.f + 63) / 64);
#define KG_NHWC_GEMM(BM, R, HALVES)                                                                                 \
  hipLaunchKernelGGL((conv2d_nhwc_kernel<Tag, BM, 64, R, HALVES>), dim3(grid, splits), dim3(convn::kThreads), 0, stream, \
                     xp, wp, y, bias, g, partial)
#define KG_NHWC_GEMM_H(BM, R) \
  if (g.halves) KG_NHWC_GEMM(BM, R, true); else KG_NHWC_GEMM(BM, R, false)
  if (bm == 128) {
    if (ring == 2) { KG_NHWC_GEMM_H(128, 2); } else { KG_NHWC_GEMM_H(128, 3); }
  } else {
    if (ring == 3) { KG_NHWC_GEMM_H(64, 3); } else { KG_NHWC_GEMM_H(64, 5); }
  }
#undef KG_NHWC_GEMM_H
#undef KG_NHWC_GEMM
}

template <typename Tag>
hipError_t launch_conv2d_nhwc(const void* x, const void* w, void* y, const void* bias, int bias_kind,
                              const ConvShape& s, const ConvNhwcPlan& plan, char* ws, hipStream_t stream) {
  using T = typename convg::IgElem<Tag>::T;
  constexpr int es = (int)sizeof(T);
  char* wpk = ws;
  char* xpk = ws + plan.w_bytes;
  float* partial = reinterpret_cast<float*>(ws + plan.w_bytes + plan.x_bytes);
  for (int n0 = 0; n0 < s.n; n0 += plan.images) {
    const int images = std::min(plan.images, s.n - n0);
    convn::Geometry g = conv_nhwc_geometry(s, images, es);
    g.bias_kind = bias_kind;
    const T* xs = static_cast<const T*>(x) + (long long)n0 * s.c * s.h * s.w;
    T* ys = static_cast<T*>(y) + (long long)n0 * s.f * g.P;
    const long long x_threads = (long long)images * g.hp * g.div_pieces.d * g.div_cpx.d;
    const long long w_chunks = n0 == 0 ? (long long)plan.w_bytes / 16 : 0;  // the weights are packed once
    const int x_blocks = (int)((x_threads + convn::kThreads - 1) / convn::kThreads);
    const int w_blocks = (int)((w_chunks + convn::kThreads - 1) / convn::kThreads);
    hipLaunchKernelGGL((conv_pack_kernel<Tag>), dim3(x_blocks + w_blocks), dim3(convn::kThreads), 0, stream, xs,
                       static_cast<const T*>(w), reinterpret_cast<u32x4*>(xpk), reinterpret_cast<u32x4*>(wpk), g, x_blocks);
    if (plan.splits > 1) g.kcs = plan.kcs;
    launch_nhwc_gemm<Tag>(xpk, wpk, ys, bias, g, plan.bm, plan.ring, plan.splits, partial, stream);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    if (plan.splits > 1) {
      const int nfp = g.NP * s.f;
      const int rgrid = (nfp + kConvReduceThreads - 1) / kConvReduceThreads;
      if (bias_kind == 0)
        hipLaunchKernelGGL((conv_splitk_reduce_kernel<Tag, 0>), dim3(rgrid), dim3(kConvReduceThreads), 0, stream,
                           partial, plan.splits, ys, bias, nfp, g.div_p, s.f);
      else if (bias_kind == 1)
        hipLaunchKernelGGL((conv_splitk_reduce_kernel<Tag, 1>), dim3(rgrid), dim3(kConvReduceThreads), 0, stream,
                           partial, plan.splits, ys, bias, nfp, g.div_p, s.f);
      else
        hipLaunchKernelGGL((conv_splitk_reduce_kernel<Tag, 2>), dim3(rgrid), dim3(kConvReduceThreads), 0, stream,
                           partial, plan.splits, ys, bias, nfp, g.div_p, s.f);
      const hipError_t e2 = hipGetLastError();
      if (e2 != hipSuccess) return e2;
    }
  }
  return hipSuccess;
}

}  // namespace kg_gfx950
