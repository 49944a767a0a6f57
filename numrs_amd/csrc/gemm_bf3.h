// Products of fp32 matrices on the bf16 matrix cores, at fp32 accuracy.
//
// An fp32 value is the sum of three bf16 values (Henry, Tang and Heinecke, "Leveraging the
// bfloat16 artificial intelligence datatype for higher-precision computations", ARITH 2019),
// x = h + m + l with h = bf16(x), m = bf16(x - h), l = x - h - m (round to nearest even; both
// differences are exact, and what is left after two roundings fits bf16's 8 bits).  Operands are split times 2^16, and
// the sums multiplied by 2^-32: every fp32 value, the subnormal ones too, is then a multiple
// of bf16's smallest subnormal, 2^-133, and the split exact (conversion and MFMA keep bf16
// subnormals: measured).  A product is
//   x y = hx hy + (hx my + mx hy) + (mx my + hx ly + lx hy) + [mx ly + lx my + lx ly],
// the bracket, at most 2^-24 |x y|, left out: six v_mfma_f32_16x16x32_bf16 per 16 x 16 x 32
// block, accumulated in fp32, smallest terms first, from zero for every 32 reduction steps;
// the sums of 32 steps are added into fp32 totals.  Measured against float64 on N(0, 1)
// operands, relative 2-norm error at R = 256 | 512 | 2048 reduction steps: 0.7 | 0.9 |
// 1.5e-7, where v_mfma_f32_32x32x2f32 with totals every 96 steps has 1.9 | 1.9 | 2.0e-7.
//
// What bounds it: gfx950's bf16 MFMA rate is 2.5 PFLOP/s against 157 TFLOP/s for fp32
// MFMAs, so six of them take 0.38 of the time at nominal rates.  The matrix units are busy
// for half of the 256 x 128 tile's cycles: a SIMD's two waves also issue 2.7 other VALU
// instructions for each MFMA (the splits, the sums of 32 steps), which takes two thirds of
// the MFMAs' time and is covered by them in part only.  On N(0, 1) data the clock is 2.1 GHz;
// on zeros, at 2.4, the same launches run 1.09 times as fast.  [4096, 2048] x [2048, 4096]
// runs at 206-209 TFLOP/s of fp32 work = 1.24 PFLOP/s of bf16 (hipBLASLt's plain bf16 product
// of that size: 1.09; the fp32 MFMA kernel that this replaced: 142 TFLOP/s).
//
// Special values.  An infinity, a NaN or a magnitude of 2^112 or more has a term x - h that
// is not finite, and makes every output of its row or column NaN or infinite; so does a sum
// of 32 products of 2^96 or more its output.  A wave that finds such an output recomputes
// its rows or columns of blocks with fp32 MFMAs, so that the results are those of fp32
// arithmetic.  One such value costs one load's latency per 32 reduction steps: 2048^3 A B^T
// 109 -> 134 us (the fp32 MFMA kernel: 131), its gradient pair with one NaN in dC 167 -> 293
// (242), 4096 x 512 -> 2048 forward 64 (66) and backward 178 (135); with four loads in flight
// in place of forty they took 425, 1205, 220 and 485.
#pragma once

#include <type_traits>

#include "common.h"

namespace bf3 {

typedef float f2 __attribute__((ext_vector_type(2)));
typedef float f4 __attribute__((ext_vector_type(4)));
// at any float's address: rows of odd length need no path of their own
typedef float f2u __attribute__((ext_vector_type(2), aligned(4)));
typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));
typedef __bf16 b2 __attribute__((ext_vector_type(2)));
typedef __bf16 b8 __attribute__((ext_vector_type(8)));
typedef uint32_t u4 __attribute__((ext_vector_type(4)));

// (a, b) -> the three terms of each, packed in pairs.
__device__ __forceinline__ void split2(float a, float b, uint32_t &h, uint32_t &m, uint32_t &l) {
  auto pack = [](float x, float y) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f2{x, y}, b2));
  };
  auto lo = [](uint32_t v) { return __builtin_bit_cast(float, v << 16); };
  auto hi = [](uint32_t v) { return __builtin_bit_cast(float, v & 0xffff0000u); };
  h = pack(a, b);
  const float ra = a - lo(h), rb = b - hi(h);
  m = pack(ra, rb);
  l = pack(ra - lo(m), rb - hi(m));
}

constexpr float kScale = 0x1p16f, kUnscale = 0x1p-32f;  // of operands, and back for their products

constexpr int kBR = 32;           // reduction steps per tile (one MFMA's)
constexpr int kChunks = kBR / 8;  // 16-byte chunks (8 bf16) of a row

// LDS image of an EXT x kBR operand tile: three planes (h, m, l) of [chunk][row] 16-byte
// chunks.  Row r of chunk ch sits at slot r ^ swizzle(ch): the 16 rows x 4 chunks of one
// MFMA operand read fall on different banks, and so do the 4 chunks x 4 rows that 16 lanes
// write when their rows are contiguous in memory.
template <int EXT>
struct Tile {
  static constexpr int kChunkStride = EXT * 16;
  static constexpr int kPlane = kChunks * kChunkStride;
  static constexpr int kBytes = 3 * kPlane;
};
__device__ __forceinline__ int swizzle(int ch) { return ((ch & 1) ? 12 : 0) ^ ((ch & 2) ? 4 : 0); }

// A thread's share of an EXT x kBR tile of an operand that is reduction-contiguous (RC:
// base[row ld + r]) or not (base[r ld + row]): N units of 8 consecutive reduction steps of
// one row.  Rows past the operand's last one read the last one (their products are not
// stored).  WIDE: 64-bit offsets, for leading dimensions of 2^24 and more.
template <bool RC, int EXT, int NT, bool WIDE>
struct Loader {
  static constexpr int N = EXT * kChunks / NT;
  static_assert(N >= 1 && N * NT == EXT * kChunks, "whole units");
  static constexpr bool kPairs = !RC && N == 2;  // two units: neighbouring rows, loaded together
  static_assert(RC || kPairs || EXT % 64 == 0, "one chunk per wave");
  using Off = typename std::conditional<WIDE, int64_t, uint32_t>::type;
  float v[N][8];
  Off off[N];   // element offset of the unit's row (and, RC, its chunk) from the tile base
  int slot[N];  // its byte offset in each plane of the LDS image

  static __device__ __forceinline__ int row(int tid, int i) {
    if (kPairs) return 2 * (tid % (EXT / 2)) + i;
    const int u = tid + NT * i;
    return RC ? u / kChunks : u % EXT;
  }
  static __device__ __forceinline__ int chunk(int tid, int i) {
    if (kPairs) return tid / (EXT / 2);
    const int u = tid + NT * i;
    return RC ? u % kChunks : u / EXT;
  }
  // The row that unit i reads, of `rows` that exist.
  static __device__ __forceinline__ int read_row(int tid, int i, int rows) {
    return kPairs ? min(row(tid, 0), rows - 2) + i : min(row(tid, i), rows - 1);
  }
  // rows: how many of the tile's rows exist; at least 1, pairs: 2 (pairs_fit).  A pair whose
  // first row is an odd last one reads the row before and that one, and trades places.
  __device__ __forceinline__ void init(int tid, int64_t ld, int rows) {
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int r = row(tid, i), from = read_row(tid, i, rows);
      const int ch = chunk(tid, i);
      const int put = kPairs && r - i > rows - 2 ? r ^ 1 : r;
      slot[i] = ch * Tile<EXT>::kChunkStride + (put ^ swizzle(ch)) * 16;
      off[i] = RC ? (Off)((Off)from * (Off)ld + (Off)(8 * ch)) : (Off)from;
    }
  }
  // Unit i (pairs: both at i = 0) of the whole tile at `base`, row 0 of the tile at its first
  // reduction step.
  __device__ __forceinline__ void load(const float *base, int64_t ld, int tid, int i) {
    if constexpr (RC) {
      const f4u a = *reinterpret_cast<const f4u *>(base + off[i]);
      const f4u b = *reinterpret_cast<const f4u *>(base + off[i] + 4);
#pragma unroll
      for (int j = 0; j < 4; ++j) v[i][j] = a[j], v[i][4 + j] = b[j];
    } else {
      const int c = __builtin_amdgcn_readfirstlane(8 * chunk(tid, i));  // one chunk per wave
      if constexpr (kPairs) {
        if (i != 0) return;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const f2u a = *reinterpret_cast<const f2u *>((base + (c + j) * ld) + off[0]);
          v[0][j] = a[0], v[1][j] = a[1];
        }
      } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) v[i][j] = (base + (c + j) * ld)[off[i]];
      }
    }
  }
  // The same for a tile of `left` <= kBR reduction steps; the others read as zero.
  __device__ __forceinline__ void load_part(const float *base, int64_t ld, int tid, int i,
                                            int left) {
    const int c = 8 * chunk(tid, i);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const bool in = c + j < left;
      const int64_t o = RC ? (int64_t)off[i] + (in ? j : -c) : (in ? (c + j) * ld : 0) + (int64_t)off[i];
      const float x = base[o];
      v[i][j] = in ? x : 0.0f;
    }
  }
  __device__ __forceinline__ float sum(int i) const {
    return ((v[i][0] + v[i][1]) + (v[i][2] + v[i][3])) + ((v[i][4] + v[i][5]) + (v[i][6] + v[i][7]));
  }
  // The terms of the values times `scale`: kScale or -kScale.
  __device__ __forceinline__ void store(char *lds, int i, float scale) const {
    u4 h, m, l;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      uint32_t a, b, c;
      split2(v[i][2 * j] * scale, v[i][2 * j + 1] * scale, a, b, c);
      h[j] = a, m[j] = b, l[j] = c;
    }
    char *p = lds + slot[i];
    *reinterpret_cast<u4 *>(p) = h;
    *reinterpret_cast<u4 *>(p + Tile<EXT>::kPlane) = m;
    *reinterpret_cast<u4 *>(p + 2 * Tile<EXT>::kPlane) = l;
  }
};

// One workgroup's output tile: WP x WQ waves of (16 BI) x (16 BJ) outputs.  Lane 16 g + c of
// a wave holds, in tot[i][j][e], row 16 i + 4 g + e and column 16 j + c of the wave's block.
template <int BI_, int BJ_, int WP_, int WQ_, bool WIDE_>
struct Shape {
  static constexpr int BI = BI_, BJ = BJ_, WP = WP_, WQ = WQ_;
  static constexpr bool WIDE = WIDE_;
  static constexpr int TP = 16 * BI * WP, TQ = 16 * BJ * WQ, NT = 64 * WP * WQ;
  static constexpr int kStage = Tile<TP>::kBytes + Tile<TQ>::kBytes;
  static constexpr int kLds = 2 * kStage;
  // Whether an operand's last tile of TP (TQ) rows has enough of them for its loader.
  static bool pairs_fit(bool rc, int64_t rows, int ext) {
    return rc || ext * kChunks / NT != 2 || rows % ext != 1;
  }
};

template <bool XRC, bool YRC, class S, bool SUMS = false>
struct Product {
  static constexpr int BI = S::BI, BJ = S::BJ, TP = S::TP, TQ = S::TQ, NT = S::NT;
  static_assert(BI % 2 == 0 && BJ % 2 == 0, "block pairs");
  using LX = Loader<XRC, TP, NT, S::WIDE>;
  f4 tot[BI][BJ];
  float rowsum[SUMS ? LX::N : 1];  // SUMS: the sums of the rows of X that the thread's units read

  // tot = X Y over R >= 1 reduction steps; X: row 0 of the tile at the first step, rows_x of
  // its TP rows exist (Y alike).  lds: S::kLds bytes.
  //
  // The MFMA's own sum rounds down rather than to nearest: its mean error is -6e-9 of the
  // result's rms whatever the sign, which sums over many outputs (a bias gradient, a
  // LayerNorm's statistics) would show (measured: 4 times the error of fp32 MFMAs in an
  // encoder block's bias gradients).  So every other tile is formed from -Y and subtracted,
  // and tiles whose `phase` differs in its last bit begin with the other sign: the mean error
  // over 64 steps is 1e-10.
  //
  // A step of the loop multiplies one LDS stage while the next one is written.  Global loads
  // run one step ahead in registers; each phase (one row block against all column blocks)
  // splits and stores one unit and issues its next load.  The one barrier stands before the
  // last phase: by then every wave has stored its share of the next stage and read its last
  // row block of this one, so the last phase's MFMAs cover the first reads of the next stage.
  __device__ __forceinline__ void run(const float *X, int64_t ldx, int rows_x, const float *Y,
                                      int64_t ldy, int rows_y, int R, int phase, char *lds) {
    using LY = Loader<YRC, TQ, NT, S::WIDE>;
    constexpr int kX = LX::N, kUnits = LX::N + LY::N;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int c = lane & 15, g = lane >> 4;
    const int at = (c ^ swizzle(g)) * 16;
    const int ax = g * Tile<TP>::kChunkStride + (wave / S::WQ) * (256 * BI) + at;
    const int by = Tile<TP>::kBytes + g * Tile<TQ>::kChunkStride + (wave % S::WQ) * (256 * BJ) + at;
    LX x;
    LY y;
    x.init(tid, ldx, rows_x);
    y.init(tid, ldy, rows_y);
    // A partial tile comes first, so that every later one is whole.
    const int nk = (R + kBR - 1) / kBR, first = R - kBR * (nk - 1);
    const int64_t xstep = XRC ? 1 : ldx, ystep = YRC ? 1 : ldy;
    auto load = [&](int u, int kt) {  // kt >= 1
      const int64_t r = first + (kt - 1) * (int64_t)kBR;
      if (u < kX)
        x.load(X + r * xstep, ldx, tid, u);
      else
        y.load(Y + r * ystep, ldy, tid, u - kX);
    };
    float part[kX] = {};  // SUMS: of up to 16 tiles
    if constexpr (SUMS)
#pragma unroll
      for (int u = 0; u < kX; ++u) rowsum[u] = 0.0f;
    // Unit u of tile kt, whose Y is negated when kt + phase is odd.
    auto store = [&](int u, int kt, char *s) {
      if (u < kX) {
        x.store(s, u, kScale);
        if constexpr (SUMS) part[u] += x.sum(u);
      } else
        y.store(s + Tile<TP>::kBytes, u - kX, ((kt + phase) & 1) ? -kScale : kScale);
    };
    // Unit u's registers are free for its next load once the units it loads with are stored.
    auto load_after = [&](int u, int kt) {
      if (LX::kPairs && u < kX) {
        if (u == kX - 1) load(0, kt);
      } else if (LY::kPairs && u >= kX) {
        if (u == kUnits - 1) load(kX, kt);
      } else {
        load(u, kt);
      }
    };
#pragma unroll
    for (int i = 0; i < BI; ++i)
#pragma unroll
      for (int j = 0; j < BJ; ++j) tot[i][j] = f4{};
#pragma unroll
    for (int u = 0; u < kX; ++u) x.load_part(X, ldx, tid, u, first);
#pragma unroll
    for (int u = 0; u < kUnits - kX; ++u) y.load_part(Y, ldy, tid, u, first);
#pragma unroll
    for (int u = 0; u < kUnits; ++u) store(u, 0, lds);
    if (nk > 1) {
#pragma unroll
      for (int u = 0; u < kUnits; ++u) load(u, 1);
    }
    __syncthreads();
    b8 a[2][3], b[BJ][3];
    auto read_a = [&](const char *s, int i) {
#pragma unroll
      for (int t = 0; t < 3; ++t)
        a[i & 1][t] = *reinterpret_cast<const b8 *>(s + ax + i * 256 + t * Tile<TP>::kPlane);
    };
    auto read_b = [&](const char *s, int j) {
#pragma unroll
      for (int t = 0; t < 3; ++t)
        b[j][t] = *reinterpret_cast<const b8 *>(s + by + j * 256 + t * Tile<TQ>::kPlane);
    };
    // Row block i against column blocks j0, j0 + 1: the small products first, from zero.
    auto pair = [&](int i, int j0, float s) {
      constexpr int kTa[6] = {2, 0, 1, 1, 0, 0}, kTb[6] = {0, 2, 1, 0, 1, 0};
      f4 t[2] = {f4{}, f4{}};
#pragma unroll
      for (int k = 0; k < 6; ++k)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          t[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i & 1][kTa[k]], b[j0 + j][kTb[k]], t[j],
                                                         0, 0, 0);
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          tot[i][j0 + j][e] = __builtin_fmaf(t[j][e], s, tot[i][j0 + j][e]);
    };
    read_a(lds, 0);
#pragma unroll
    for (int j = 0; j < BJ; ++j) read_b(lds, j);
    auto step = [&](int kt, auto more_t) {
      constexpr bool kMore = decltype(more_t)::value;
      const char *cur = lds + (kt & 1) * S::kStage;
      char *nxt = lds + ((kt + 1) & 1) * S::kStage;
      const float s = ((kt + phase) & 1) ? -kUnscale : kUnscale;
      const int later = min(kt + 2, nk - 1);  // past the end: the last tile again, unused
#pragma unroll
      for (int i = 0; i + 1 < BI; ++i) {
        read_a(cur, i + 1);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (kMore) {
#pragma unroll
          for (int u = 0; u < kUnits; ++u)
            if (u * (BI - 1) / kUnits == i) {
              store(u, kt + 1, nxt);
              load_after(u, later);
            }
        }
#pragma unroll
        for (int j = 0; j < BJ; j += 2) pair(i, j, s);
        __builtin_amdgcn_sched_barrier(0);
      }
      if constexpr (kMore) {
        __syncthreads();
        read_a(nxt, 0);  // BI is even: the buffer that the last row block does not use
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int j = 0; j < BJ; j += 2) {
        pair(BI - 1, j, s);
        if constexpr (kMore) {
          __builtin_amdgcn_sched_barrier(0);
          read_b(nxt, j);
          read_b(nxt, j + 1);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    };
    for (int kt = 0; kt + 1 < nk; ++kt) {
      step(kt, std::true_type{});
      if constexpr (SUMS)
        if ((kt & 15) == 14)
#pragma unroll
          for (int u = 0; u < kX; ++u) rowsum[u] += part[u], part[u] = 0.0f;
    }
    if constexpr (SUMS)
#pragma unroll
      for (int u = 0; u < kX; ++u) rowsum[u] += part[u];
    step(nk - 1, std::false_type{});
    f4 z = {};  // x 0 is NaN where an output x is not finite
#pragma unroll
    for (int i = 0; i < BI; ++i)
#pragma unroll
      for (int j = 0; j < BJ; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) z[e] = __builtin_fmaf(tot[i][j][e], 0.0f, z[e]);
    const bool bad = !((z[0] + z[1]) + (z[2] + z[3]) == 0.0f);
    if (__any(bad)) fp32(X, ldx, rows_x, Y, ldy, rows_y, R);
  }

  // The rows of the wave's 16 x 16 blocks that hold an output that is not finite, or the columns
  // where those are fewer, again with fp32 MFMAs straight from global memory (see "Special
  // values"): v_mfma_f32_16x16x4f32, lane (g, c) feeding row or column c at reduction step
  // 16 s + 4 g + j to MFMA j of 16 steps; sums of 32 steps, whose loads are all issued before the
  // first MFMA, added into the totals.  Few waves do this, so that a load's latency per 32 steps
  // and line of blocks is what it costs.  A line at a time keeps it within the product's registers.
  __device__ __forceinline__ void fp32(const float *X, int64_t ldx, int rows_x, const float *Y,
                                       int64_t ldy, int rows_y, int R) {
    using Off = typename std::conditional<S::WIDE, int64_t, uint32_t>::type;
    unsigned rows = 0, cols = 0;
#pragma unroll
    for (int i = 0; i < BI; ++i)
#pragma unroll
      for (int j = 0; j < BJ; ++j) {
        const f4 z = tot[i][j] * 0.0f;
        if (__any(!((z[0] + z[1]) + (z[2] + z[3]) == 0.0f))) rows |= 1u << i, cols |= 1u << j;
      }
    // Steps k + 4 g .. + 3 of the row whose step 0 is at element `off`.
    auto load = [&](auto rc, float (&v)[4], const float *base, int64_t ld, Off off, int g, int k) {
      if constexpr (decltype(rc)::value) {
        const f4u a = *reinterpret_cast<const f4u *>(base + k + (off + (Off)(4 * g)));
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = a[j];
      } else {
        const Off at = off + (Off)(4 * g) * (Off)ld;
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = (base + (k + j) * ld)[at];
      }
    };
    // Line l of blocks: row l of X's against all of Y's, or column l of Y's against all of X's.
    auto line = [&](auto row_t, int l, auto &&tot_of) {
      constexpr bool ROW = decltype(row_t)::value;
      constexpr int N = ROW ? BJ : BI;
      int tid = threadIdx.x;
      asm volatile("" : "+v"(tid));  // lane values are not kept from the product or the last line
      const int lane = tid & 63, wave = tid >> 6;
      const int c = lane & 15, g = lane >> 4;
      auto off_x = [&](int b) {
        const Off r = (Off)min((wave / S::WQ) * (16 * BI) + 16 * b + c, rows_x - 1);
        return XRC ? r * (Off)ldx : r;
      };
      auto off_y = [&](int b) {
        const Off r = (Off)min((wave % S::WQ) * (16 * BJ) + 16 * b + c, rows_y - 1);
        return YRC ? r * (Off)ldy : r;
      };
      const Off off = ROW ? off_x(l) : off_y(l);
      using One = std::integral_constant<bool, ROW ? XRC : YRC>;
      using All = std::integral_constant<bool, ROW ? YRC : XRC>;
      const float *const A = ROW ? X : Y, *const B = ROW ? Y : X;
      const int64_t lda = ROW ? ldx : ldy, ldb = ROW ? ldy : ldx;
      auto mfma = [&](float one, float other, f4 t) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(ROW ? one : other, ROW ? other : one, t, 0, 0, 0);
      };
      Off all[N];
      f4 t[N];
#pragma unroll
      for (int n = 0; n < N; ++n) {
        all[n] = ROW ? off_y(n) : off_x(n);
        tot_of(n) = t[n] = f4{};
      }
      int r0 = 0;
#pragma unroll 1
      for (; r0 + 32 <= R; r0 += 32) {
        float a[2][4], b[2][N][4];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          load(One{}, a[u], A, lda, off, g, r0 + 16 * u);
#pragma unroll
          for (int n = 0; n < N; ++n) load(All{}, b[u][n], B, ldb, all[n], g, r0 + 16 * u);
        }
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
          for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int n = 0; n < N; ++n) t[n] = mfma(a[u][e], b[u][n][e], t[n]);
#pragma unroll
        for (int n = 0; n < N; ++n) tot_of(n) += t[n], t[n] = f4{};
      }
#pragma unroll 1
      for (; r0 < R; r0 += 4) {  // fewer than 32 steps: step r0 + g
        const bool in = r0 + g < R;
        const int64_t r = in ? r0 + g : 0;
        const float a = A[(int64_t)off + (One::value ? r : r * lda)];
#pragma unroll
        for (int n = 0; n < N; ++n) {
          const float b = B[(int64_t)all[n] + (All::value ? r : r * ldb)];
          t[n] = mfma(in ? a : 0.0f, in ? b : 0.0f, t[n]);
        }
      }
#pragma unroll
      for (int n = 0; n < N; ++n) tot_of(n) += t[n];
    };
    if (__builtin_popcount(rows) <= __builtin_popcount(cols)) {
#pragma unroll
      for (int i = 0; i < BI; ++i)
        if (rows >> i & 1) line(std::true_type{}, i, [&](int n) -> f4 & { return tot[i][n]; });
    } else {
#pragma unroll
      for (int j = 0; j < BJ; ++j)
        if (cols >> j & 1) line(std::false_type{}, j, [&](int n) -> f4 & { return tot[n][j]; });
    }
  }
};

}  // namespace bf3
