// Attention on the bf16 matrix cores at fp32 accuracy (the three-term splits of gemm_bf3.h),
// for head sizes that are multiples of 8 up to 128 and any sequence length.
//
//   forward        P = softmax(alpha Q K^T) stored, O = P V
//   query rows     D = dO . O, dS = P (dO V^T - D), dQ = alpha dS K
//   key rows       dV = P^T dO, dK = alpha dS^T Q, with dS formed again from P, dO V^T and D
// (the two in one launch where they are few)
//
// A wave owns 16 rows (of queries, or keys in the last kernel) as the columns c of its MFMAs;
// the workgroup walks the other sequence in blocks of BLK rows staged in LDS.  The first
// product of a block leaves lane (g, c) with rows 16 k + 4 g + e (e = 0..3) against its own
// row: exactly 8 values per 32 rows, which are split in registers and are the second operand
// of the second product.  That product's reduction runs over the rows in the order (g, [16
// k + 4 g + e]), and the transposed LDS images hold their rows in that order, so nothing of S
// x S size passes through LDS, and neither S nor dS is written to memory.
//
// The forward walks the keys twice (row maxima and sums, then P and O), since P is stored
// normalised; one more product in place of a pass over P.
#pragma once

#include "gemm_bf3.h"

namespace attn {

using bf3::b8;
using bf3::f4;
using bf3::f4u;
using bf3::kScale;
using bf3::kUnscale;
using bf3::u4;

// NW x NG waves: wave w owns rows 16 (w % NW) .. + 15 of the workgroup's 16 NW against part
// w / NW of every staged block: eight row groups where their workgroups fill the chip, else
// four with the staged rows halved between two sets of waves.
template <int DH_, int NW_, int NG_>
struct Cfg {
  static constexpr int DH = DH_, NW = NW_, NG = NG_, NT = 64 * NW * NG;  // DH: the head size rounded up to 32
  static constexpr int SUB = DH <= 64 ? 64 : 32, N16 = SUB / 16;         // a wave's staged rows per step
  static constexpr int BLK = SUB * NG;                                   // all of them
  static constexpr int NS = DH / 32, NB = DH / 16;                       // reduction steps, output blocks
  static constexpr int kPlane = BLK * DH * 2;                            // bytes of one term's image
  static constexpr int kImage = 3 * kPlane;
  static constexpr int kUnits = (BLK * DH / 8 + NT - 1) / NT;
  // A wave's f4[NB] of every group but the first fit in `images` images.
  static constexpr bool parts_fit(int images) { return (NG - 1) * NW * 64 * NB * 16 <= images * kImage; }
};

// The terms of operands, which come multiplied by kScale (products: times kUnscale).
__device__ __forceinline__ void split8(const float (&v)[8], u4 &h, u4 &m, u4 &l) {
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    uint32_t a, b, c;
    bf3::split2(v[2 * j], v[2 * j + 1], a, b, c);
    h[j] = a, m[j] = b, l[j] = c;
  }
}

struct Terms {
  b8 t[3];
  __device__ __forceinline__ void set(const float (&v)[8]) {
    u4 h, m, l;
    split8(v, h, m, l);
    t[0] = __builtin_bit_cast(b8, h), t[1] = __builtin_bit_cast(b8, m), t[2] = __builtin_bit_cast(b8, l);
  }
};

// acc[i] += a[i] b[i] for N independent sums in turn, the small products first: the sums
// cover each other's MFMA latency.
template <int N>
__device__ __forceinline__ void mma(f4 (&acc)[N], const Terms (&a)[N], const Terms *const (&b)[N]) {
  constexpr int kTa[6] = {2, 0, 1, 1, 0, 0}, kTb[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
  for (int k = 0; k < 6; ++k)
#pragma unroll
    for (int i = 0; i < N; ++i)
      acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i].t[kTa[k]], b[i]->t[kTb[k]], acc[i], 0, 0, 0);
}

// A thread's share of a BLK x DH block of a matrix (rows r0 .. of `n`, row stride ld, dh
// columns, the others zero; rows past the last read the last), and its LDS image.
//   !TR: a unit is 8 consecutive columns of a row; image [plane][column chunk][row].
//    TR: a unit is one column of 8 rows, those of chunk g of 32 rows being 4 g .. 4 g + 3 and
//        16 + 4 g .. + 3; image [plane][row group, chunk][column].
// Slots are swizzled as in bf3::Tile.
template <class C, bool TR>
struct Block {
  float v[C::kUnits][8];
  int off[C::kUnits];  // element offset of the unit's first row and column in a block
  bool in[C::kUnits];  // its columns exist
  static __device__ __forceinline__ bool live(int u) {
    return C::BLK * C::DH / 8 % C::NT == 0 || u < C::BLK * C::DH / 8;
  }
  static __device__ __forceinline__ int row(int u) {
    return TR ? 32 * (u / C::DH >> 2) + 4 * (u / C::DH & 3) : u / (C::DH / 8);
  }
  static __device__ __forceinline__ int col(int u) { return TR ? u % C::DH : 8 * (u % (C::DH / 8)); }
  __device__ __forceinline__ void init(int ld, int dh, int tid) {
#pragma unroll
    for (int i = 0; i < C::kUnits; ++i) {
      const int u = tid + C::NT * i;
      in[i] = live(u) && col(u) < dh;
      off[i] = in[i] ? row(u) * ld + col(u) : 0;
    }
  }
  // Block starting at row r0 of n.
  __device__ __forceinline__ void load(const float *base, int ld, int r0, int n, int tid) {
    const float *p0 = base + (int64_t)r0 * ld;
    const bool whole = r0 + C::BLK <= n;
#pragma unroll
    for (int i = 0; i < C::kUnits; ++i) {
      if constexpr (TR) {
        if (whole) {
#pragma unroll
          for (int j = 0; j < 8; ++j) v[i][j] = (p0 + ((j & 3) + 16 * (j >> 2)) * ld)[off[i]];
        } else {
          const int u = tid + C::NT * i, left = n - 1 - r0;
          const int d = in[i] ? col(u) : 0;
#pragma unroll
          for (int j = 0; j < 8; ++j) v[i][j] = p0[min(row(u) + (j & 3) + 16 * (j >> 2), left) * ld + d];
        }
      } else {
        const int u = tid + C::NT * i;
        const float *p = p0 + (whole ? off[i] : min(row(u), n - 1 - r0) * ld + (in[i] ? col(u) : 0));
        const f4u a = *reinterpret_cast<const f4u *>(p), b = *reinterpret_cast<const f4u *>(p + 4);
#pragma unroll
        for (int j = 0; j < 4; ++j) v[i][j] = a[j], v[i][4 + j] = b[j];
      }
    }
  }
  __device__ __forceinline__ void store(char *lds, int tid) const {
#pragma unroll
    for (int i = 0; i < C::kUnits; ++i) {
      const int u = tid + C::NT * i;
      if (!live(u)) continue;
      constexpr int kRow = TR ? C::DH : C::BLK;
      const int slot = TR ? u % C::DH : u / (C::DH / 8), ch = TR ? u / C::DH : u % (C::DH / 8);
      char *p = lds + ((int64_t)ch * kRow + (slot ^ bf3::swizzle(ch & 3))) * 16;
      float x[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) x[j] = v[i][j] * kScale;
      u4 h, m, l;
      split8(x, h, m, l);
      if (!in[i]) h = m = l = u4{};  // a column past the head's last
      *reinterpret_cast<u4 *>(p) = h;
      *reinterpret_cast<u4 *>(p + C::kPlane) = m;
      *reinterpret_cast<u4 *>(p + 2 * C::kPlane) = l;
    }
  }
};

// First-operand fragment: 16 slots from `slot0` of chunk 4 step + g.
template <class C, bool TR>
__device__ __forceinline__ void frag(Terms &f, const char *lds, int step, int slot0, int c, int g) {
  constexpr int kRow = TR ? C::DH : C::BLK;
  const char *p = lds + ((4 * step + g) * kRow + slot0 + (c ^ bf3::swizzle(g))) * 16;
#pragma unroll
  for (int t = 0; t < 3; ++t) f.t[t] = *reinterpret_cast<const b8 *>(p + t * C::kPlane);
}

// The wave's own rows as second operand: lane (g, c) holds row `row`, columns 32 s + 8 g .. + 7;
// times kScale, odd steps negated (blocks32 subtracts them).
template <class C>
__device__ __forceinline__ void own_rows(Terms (&f)[C::NS], const float *row, int dh, int g) {
#pragma unroll
  for (int s = 0; s < C::NS; ++s) {
    const int at = 32 * s + 8 * g;
    const bool in = at < dh;
    const float *p = row + (in ? at : 0);
    const f4u a = *reinterpret_cast<const f4u *>(p), b = *reinterpret_cast<const f4u *>(p + 4);
    const float scale = (s & 1) ? -kScale : kScale;
    float v[8];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      v[j] = in ? scale * a[j] : 0.0f;
      v[4 + j] = in ? scale * b[j] : 0.0f;
    }
    f[s].set(v);
  }
}

// y[u] kUnscale: the staged rows 16 (k + u) + 4 g + e against the wave's row c, u = 0, 1.
// Steps alternate in sign: the MFMA's sums round down (gemm_bf3.h).
template <class C>
__device__ __forceinline__ void blocks32(f4 (&y)[2], const char *lds, int k, const Terms (&own)[C::NS], int c,
                                         int g) {
  f4 odd[2] = {f4{}, f4{}};
  y[0] = y[1] = f4{};
#pragma unroll
  for (int s = 0; s < C::NS; s += 2) {
    if (s + 1 < C::NS) {
      Terms a[4];
      f4 t[4] = {y[0], y[1], odd[0], odd[1]};
#pragma unroll
      for (int u = 0; u < 4; ++u) frag<C, false>(a[u], lds, s + (u >> 1), 16 * (k + (u & 1)), c, g);
      const Terms *const b[4] = {&own[s], &own[s], &own[s + 1 < C::NS ? s + 1 : s], &own[s + 1 < C::NS ? s + 1 : s]};
      mma(t, a, b);
      y[0] = t[0], y[1] = t[1], odd[0] = t[2], odd[1] = t[3];
    } else {
      Terms a[2];
#pragma unroll
      for (int u = 0; u < 2; ++u) frag<C, false>(a[u], lds, s, 16 * (k + u), c, g);
      const Terms *const b[2] = {&own[s], &own[s]};
      mma(y, a, b);
    }
  }
#pragma unroll
  for (int u = 0; u < 2; ++u) y[u] -= odd[u];
}

// acc[b] += sign (the image's columns 16 b + 4 g + e) of 32 staged rows times the wave's values p
// (times kScale).
template <class C>
__device__ __forceinline__ void rows32(f4 (&acc)[C::NB], const char *lds, int grp, const Terms &p,
                                       float sign, int c, int g) {
#pragma unroll
  for (int b = 0; b < C::NB; b += 2) {
    Terms a[2];
    f4 t[2] = {f4{}, f4{}};
#pragma unroll
    for (int u = 0; u < 2; ++u) frag<C, true>(a[u], lds, grp, 16 * (b + u), c, g);
    const Terms *const q[2] = {&p, &p};
    mma(t, a, q);
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[b + u][e] = __builtin_fmaf(t[u][e], sign * kUnscale, acc[b + u][e]);
  }
}

// Whether any value of the wave's live rows is not finite.
template <int N>
__device__ __forceinline__ bool any_bad(const f4 (&acc)[N], bool live) {
  float z = 0.0f;
#pragma unroll
  for (int b = 0; b < N; ++b)
#pragma unroll
    for (int e = 0; e < 4; ++e) z = __builtin_fmaf(acc[b][e], 0.0f, z);
  return __any(live && !(z == 0.0f));
}

// 4 values of row `p` from `at`, zero from `n` on (whole: none are).
__device__ __forceinline__ f4 load4(const float *p, int at, int n, bool whole) {
  if (whole || at + 4 <= n) {
    const f4u v = *reinterpret_cast<const f4u *>(p + at);
    return f4{v[0], v[1], v[2], v[3]};
  }
  f4 v = {};
#pragma unroll
  for (int e = 0; e < 4; ++e)
    if (at + e < n) v[e] = p[at + e];
  return v;
}

// Head z's columns of the wave's row: lane (g, c) writes (add: adds) 16 b + 4 g .. + 3 times `alpha`.
template <class C>
__device__ __forceinline__ void store_rows(float *row, const f4 (&acc)[C::NB], float alpha, int dh, int g, int add) {
#pragma unroll
  for (int b = 0; b < C::NB; ++b)
    if (16 * b + 4 * g < dh) {
      f4u *at = reinterpret_cast<f4u *>(row + 16 * b + 4 * g);
      f4u v;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = alpha * acc[b][e];
      *at = add ? *at + v : v;
    }
}

// fp32 forms of blocks32 and rows32 from global memory (non-finite values, see gemm_bf3.h), for
// 16 N rows at a time; the caller issues a step's loads before it uses any.  With one NaN among
// 16 x 256 x 8 x 64 the forward takes 24 -> 79 us and the backward 48 -> 180 (134 and 310 with
// 16 rows at a time and each column's load before its MFMA).
template <class C>
struct Fp32 {
  static constexpr int N = C::DH <= 64 ? 2 : 1, ROWS = 16 * N;
  float own[C::NB][4];  // the wave's row: columns 16 b + 4 g + j
  __device__ __forceinline__ void set(const float *row, int dh, int g) {
#pragma unroll
    for (int b = 0; b < C::NB; ++b) load(own[b], row, 16 * b + 4 * g, dh);
  }
  static __device__ __forceinline__ void load(float (&v)[4], const float *row, int at, int dh) {
    const bool in = at < dh;  // dh is a multiple of 8
    const f4u a = *reinterpret_cast<const f4u *>(row + (in ? at : 0));
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = in ? a[j] : 0.0f;
  }
  // Rows r0 + 16 u + c of n of `x`, columns 16 b + 4 g + j (past the last: the last row).
  struct Rows {
    float v[N][C::NB][4];
    __device__ __forceinline__ void load(const float *x, int64_t ld, int r0, int n, int dh, int c, int g) {
#pragma unroll
      for (int u = 0; u < N; ++u)
#pragma unroll
        for (int b = 0; b < C::NB; ++b)
          Fp32::load(v[u][b], x + (int64_t)min(r0 + 16 * u + c, n - 1) * ld, 16 * b + 4 * g, dh);
    }
  };
  // Rows r0 + 16 u + 4 g + e of n of `x`, columns 16 b + c; zero past the last.
  struct Cols {
    float v[N][4][C::NB];
    __device__ __forceinline__ void load(const float *x, int64_t ld, int r0, int n, int dh, int c, int g) {
#pragma unroll
      for (int u = 0; u < N; ++u)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int r = r0 + 16 * u + 4 * g + e;
          const float *xr = x + (int64_t)min(r, n - 1) * ld;
#pragma unroll
          for (int b = 0; b < C::NB; ++b) {
            const int d = 16 * b + c;
            const float w = xr[d < dh ? d : 0];
            v[u][e][b] = r < n && d < dh ? w : 0.0f;
          }
        }
    }
  };
  // y[u]: rows r0 + 16 u + 4 g + e against the wave's row.
  __device__ __forceinline__ void dots(f4 (&y)[N], const Rows &x) const {
#pragma unroll
    for (int u = 0; u < N; ++u) y[u] = f4{};
#pragma unroll
    for (int b = 0; b < C::NB; ++b)
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int u = 0; u < N; ++u)
          y[u] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.v[u][b][j], own[b][j], y[u], 0, 0, 0);
  }
  // acc[b] += columns 16 b + 4 g + e of the rows times the wave's values p.
  static __device__ __forceinline__ void add(f4 (&acc)[C::NB], const Cols &x, const f4 (&p)[N]) {
#pragma unroll
    for (int u = 0; u < N; ++u)
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int b = 0; b < C::NB; ++b)
          acc[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.v[u][e][b], p[u][e], acc[b], 0, 0, 0);
  }
};

// The workgroup's head z and first row: XCD k (hardware ids k, k + 8, ...) owns a contiguous
// run of heads, whose workgroups stage the same rows through one L2.
__device__ __forceinline__ void place(int &z, int &blk) {
  const int nx = gridDim.x, nb = nx * gridDim.y, lin = blockIdx.x + nx * blockIdx.y;
  const int xcd = lin & 7, per = nb >> 3, more = nb & 7;
  const int logical = xcd * per + min(xcd, more) + (lin >> 3);
  z = logical / nx;
  blk = logical - z * nx;
}

// Blocks 0 .. nb - 1 through the workgroup's LDS images: load(i) global rows to registers,
// store() them, use(i).  MOST > 0: nb is at most MOST and the blocks are unrolled.
template <int MOST, class Load, class Store, class Use>
__device__ __forceinline__ void walk(int nb, Load load, Store store, Use use) {
  auto body = [&](int i) {
    __syncthreads();  // the last block's reads
    store();
    if (i + 1 < nb) load(i + 1);
    __syncthreads();
    use(i);
  };
  load(0);
  if constexpr (MOST > 0) {
#pragma unroll
    for (int i = 0; i < MOST; ++i)
      if (i < nb) body(i);
  } else {
    for (int i = 0; i < nb; ++i) body(i);
  }
}

// acc summed over the groups' waves, in the first group's.  lds: the images, free.
template <class C>
__device__ __forceinline__ void join_groups(f4 (&acc)[C::NB], char *lds, int wave, int lane) {
  if constexpr (C::NG > 1) {
    f4 *part = reinterpret_cast<f4 *>(lds);
    const int grp = wave / C::NW, rows = wave % C::NW;
    __syncthreads();
    if (grp > 0)
#pragma unroll
      for (int b = 0; b < C::NB; ++b) part[(((grp - 1) * C::NW + rows) * C::NB + b) * 64 + lane] = acc[b];
    __syncthreads();
    if (grp == 0)
#pragma unroll
      for (int n = 0; n + 1 < C::NG; ++n)
#pragma unroll
        for (int b = 0; b < C::NB; ++b) acc[b] += part[((n * C::NW + rows) * C::NB + b) * 64 + lane];
  }
}

// A row's scores in base 2, y (alpha log2 e) in two parts so that the constant's rounding
// does not scale with the score, less the row's reference m.
struct Scale {
  float hi, lo;
  // INF: y may be -inf (a probability of 0), which the two-part product would make NaN
  template <bool INF>
  __device__ __forceinline__ float at(float y, float m) const {
    const float t = __builtin_fmaf(y, hi, -m);
    return INF && y == -INFINITY ? t : __builtin_fmaf(y, lo, t);
  }
};

// Running maximum and sum of 2^score of one lane's keys.
struct RowStat {
  float m = -INFINITY, l = 0.0f;
  // Keys key0 + 16 k + e, those from S on left out (WHOLE: there are none).  INF, the pass whose
  // result stands: a NaN score makes the row's sum NaN, also where fmaxf drops it because the
  // lane has no other key yet.  (In the other form such a key's own probability is NaN, and with
  // it the row's output, which calls for this pass.)
  template <bool INF, bool WHOLE, int N>
  __device__ __forceinline__ void add(const f4 (&y)[N], const Scale &sc, int key0, int S) {
    float top = -INFINITY;
    bool nan = false;
#pragma unroll
    for (int k = 0; k < N; ++k)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (WHOLE || key0 + 16 * k + e < S) {
          top = fmaxf(top, y[k][e]);
          nan = nan || y[k][e] != y[k][e];
        }
    if (INF && nan) {
      l = NAN;
      m = fmaxf(m, 0.0f);  // not -inf: part() keeps l
      return;
    }
    top = fmaxf(m, top * sc.hi);
    if (top == -INFINITY) return;  // no key of this lane yet
    l = l * __builtin_amdgcn_exp2f(m - top);
    m = top;
    float part = 0.0f;  // a block's own sum: fewer roundings at l's size
#pragma unroll
    for (int k = 0; k < N; ++k)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (WHOLE || key0 + 16 * k + e < S) part += __builtin_amdgcn_exp2f(sc.at<INF>(y[k][e], m));
    l += part;
  }
  __device__ __forceinline__ static float part(float l, float m, float top) {
    return m == -INFINITY ? 0.0f : l * __builtin_amdgcn_exp2f(m - top);
  }
  // over the row's four lanes
  __device__ __forceinline__ void join() {
    const float top = rows4(m, [](float a, float b) { return fmaxf(a, b); });
    l = rows4(part(l, m, top), [](float a, float b) { return a + b; });
    m = top;
  }
  // over the groups' waves too; lds: two floats per row and group
  template <class C>
  __device__ __forceinline__ void join_groups(float *lds, int wave, int lane) {
    if constexpr (C::NG > 1) {
      const int row = wave % C::NW * 16 + (lane & 15);
      if (lane < 16) {
        lds[(wave / C::NW * 2) * 16 * C::NW + row] = m;
        lds[(wave / C::NW * 2 + 1) * 16 * C::NW + row] = l;
      }
      __syncthreads();
      float ms[C::NG], top = -INFINITY, sum = 0.0f;
#pragma unroll
      for (int n = 0; n < C::NG; ++n) {
        ms[n] = lds[2 * n * 16 * C::NW + row];
        top = fmaxf(top, ms[n]);
      }
#pragma unroll
      for (int n = 0; n < C::NG; ++n) sum += part(lds[(2 * n + 1) * 16 * C::NW + row], ms[n], top);
      m = top;
      l = sum;
    }
  }
};

// KEEP: the scores of up to KEEP blocks (all of them) stay in registers between the two walks.
template <class C, int KEEP>
__global__ void __launch_bounds__(C::NT) fwd_kernel(const float *q, const float *k, const float *v, int ld,
                                                    float *P, float *out, int64_t ldo, int S, int H, int dh,
                                                    Scale sc) {
  __shared__ __attribute__((aligned(1024))) char lds[2 * C::kImage];
  __shared__ float rowstat[2 * C::NG * 16 * C::NW];
  static_assert(C::parts_fit(2), "partial outputs");
  char *const kl = lds, *const vl = lds + C::kImage;
  constexpr int N16 = C::N16;
  int z, blk;
  place(z, blk);
  const int tid = threadIdx.x, lane = tid & 63, c = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), grp = wave / C::NW, n0 = grp * N16;
  const int row = blk * 16 * C::NW + wave % C::NW * 16 + c;
  const bool live = row < S;
  const int64_t at = (int64_t)(z / H) * S * ld + (z % H) * dh;
  q += at + (int64_t)min(row, S - 1) * ld;
  k += at;
  v += at;
  Terms own[C::NS];
  own_rows<C>(own, q, dh, g);
  Block<C, false> kb;
  Block<C, true> vb;
  kb.init(ld, dh, tid);
  vb.init(ld, dh, tid);
  const int nb = (S + C::BLK - 1) / C::BLK;
  RowStat st;
  const Scale sf{sc.hi * kUnscale, sc.lo * kUnscale};  // of blocks32's scores
  f4 kept[KEEP > 0 ? KEEP : 1][N16];
  // The wave's first key of block i, and whether all of its keys there exist.
  auto first = [&](int i) { return i * C::BLK + grp * C::SUB; };
  auto whole = [&](int i) { return first(i) + C::SUB <= S; };
  auto stat = [&](int i, f4 (&y)[N16]) {
#pragma unroll
    for (int n = 0; n < N16; n += 2) {
      f4 t[2];
      blocks32<C>(t, kl, n0 + n, own, c, g);
      y[n] = t[0], y[n + 1] = t[1];
    }
    if (whole(i))
      st.add<false, true>(y, sf, first(i) + 4 * g, S);
    else
      st.add<false, false>(y, sf, first(i) + 4 * g, S);
  };
  auto load_k = [&](int i) { kb.load(k, ld, i * C::BLK, S, tid); };
  walk<KEEP>(nb, load_k, [&]() { kb.store(kl, tid); }, [&](int i) {
    if constexpr (KEEP > 0) {
      stat(i, kept[i]);
    } else {
      f4 y[N16];
      stat(i, y);
    }
  });
  st.join();
  st.join_groups<C>(rowstat, wave, lane);
  float inv = 1.0f / st.l;
  f4 acc[C::NB];
#pragma unroll
  for (int b = 0; b < C::NB; ++b) acc[b] = f4{};
  float *Pr = P + ((int64_t)z * S + min(row, S - 1)) * S;
  // Keys 16 n .. 16 n + 31 of block i, scores y: their probabilities, stored and multiplied by V.
  auto finish = [&](auto whole_t, int i, int n, const f4 (&y)[2]) {
    constexpr bool WHOLE = decltype(whole_t)::value;
    const float sign = (i * (C::SUB / 32) + n / 2) & 1 ? -1.0f : 1.0f;
    float p[8];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int key = first(i) + 16 * (n + u) + 4 * g;
      f4u w;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        w[e] = __builtin_amdgcn_exp2f(sf.at<false>(y[u][e], st.m)) * inv;
        if (!WHOLE && key + e >= S) w[e] = 0.0f;
        p[4 * u + e] = sign * kScale * w[e];
      }
      if (live && (WHOLE || key + 4 <= S))
        *reinterpret_cast<f4u *>(Pr + key) = w;
      else if (live)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (key + e < S) Pr[key + e] = w[e];
    }
    Terms pt;
    pt.set(p);
    rows32<C>(acc, vl, (n0 + n) / 2, pt, sign, c, g);
  };
  walk<KEEP>(
      nb,
      [&](int i) {
        if (KEEP == 0) load_k(i);
        vb.load(v, ld, i * C::BLK, S, tid);
      },
      [&]() {
        if (KEEP == 0) kb.store(kl, tid);
        vb.store(vl, tid);
      },
      [&](int i) {
        const bool all = whole(i);
#pragma unroll
        for (int n = 0; n < N16; n += 2) {
          f4 t[2];
          if constexpr (KEEP > 0)
            t[0] = kept[i][n], t[1] = kept[i][n + 1];
          else
            blocks32<C>(t, kl, n0 + n, own, c, g);
          if (all)
            finish(std::true_type{}, i, n, t);
          else
            finish(std::false_type{}, i, n, t);
        }
      });
  join_groups<C>(acc, lds, wave, lane);
  if (grp > 0) return;
  if (any_bad(acc, live)) {  // again in fp32, from global memory
    using F = Fp32<C>;
    F f;
    f.set(q, dh, g);
    st = RowStat{};
    for (int r0 = 0; r0 < S; r0 += F::ROWS) {
      typename F::Rows kr;
      kr.load(k, ld, r0, S, dh, c, g);
      f4 y[F::N];
      f.dots(y, kr);
      st.add<true, false>(y, sc, r0 + 4 * g, S);
    }
    st.join();
    inv = 1.0f / st.l;
#pragma unroll
    for (int b = 0; b < C::NB; ++b) acc[b] = f4{};
    for (int r0 = 0; r0 < S; r0 += F::ROWS) {
      typename F::Rows kr;
      typename F::Cols vr;
      kr.load(k, ld, r0, S, dh, c, g);
      vr.load(v, ld, r0, S, dh, c, g);
      f4 y[F::N], p[F::N];
      f.dots(y, kr);
#pragma unroll
      for (int u = 0; u < F::N; ++u)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int key = r0 + 16 * u + 4 * g + e;
          p[u][e] = key < S ? __builtin_amdgcn_exp2f(sc.at<true>(y[u][e], st.m)) * inv : 0.0f;
          if (live && key < S) Pr[key] = p[u][e];
        }
      F::add(acc, vr, p);
    }
  }
  if (live) store_rows<C>(out + ((int64_t)(z / H) * S + row) * ldo + (z % H) * dh, acc, 1.0f, dh, g, 0);
}

// D[z, row], the softmax backward's row total of P dP, and dQ (null: D alone).  D comes from a walk
// over the keys of its own, from the forward's output, D = dO . (P V) = dO . O, or is given.
// Workgroup blk of head z; lds: two images.
enum { kWalkD, kOutD, kGivenD };
template <class C, int MODE>
__device__ __forceinline__ void bwd_query(char *lds, int z, int blk, const float *k, const float *v, int ld,
                                          const float *P, const float *dout, const float *out, int64_t ldo,
                                          float *D, float *dq, int S, int H, int dh, float alpha, int add) {
  static_assert(C::parts_fit(2), "partial outputs");
  char *const vl = lds, *const kl = lds + C::kImage;
  constexpr int N16 = C::N16;
  const int tid = threadIdx.x, lane = tid & 63, c = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), grp = wave / C::NW, n0 = grp * N16;
  const int row = blk * 16 * C::NW + wave % C::NW * 16 + c;
  const bool live = row < S;
  const int rc = min(row, S - 1);
  const int64_t at = (int64_t)(z / H) * S * ld + (z % H) * dh;
  const int64_t ato = ((int64_t)(z / H) * S + rc) * ldo + (z % H) * dh;
  k += at;
  v += at;
  Terms own[C::NS];
  own_rows<C>(own, dout + ato, dh, g);
  const float *Pr = P + ((int64_t)z * S + rc) * S;
  Block<C, false> vb;
  Block<C, true> kb;
  const int nb = (S + C::BLK - 1) / C::BLK;
  f4 acc[C::NB];
#pragma unroll
  for (int b = 0; b < C::NB; ++b) acc[b] = f4{};
  vb.init(ld, dh, tid);
  kb.init(ld, dh, tid);
  auto first = [&](int i) { return i * C::BLK + grp * C::SUB; };
  f4 p[N16];
  int next = 0;
  auto load_p = [&](int i) {
#pragma unroll
    for (int n = 0; n < N16; ++n) p[n] = load4(Pr, first(i) + 16 * n + 4 * g, S, first(i) + C::SUB <= S);
  };
  float d = 0.0f;
  if constexpr (MODE == kGivenD) {
    d = D[(int64_t)z * S + rc];
  } else if constexpr (MODE == kOutD) {
#pragma unroll
    for (int s = 0; s < C::NS; ++s)
      if (32 * s + 8 * g < dh)
#pragma unroll
        for (int j = 0; j < 8; ++j) d += dout[ato + 32 * s + 8 * g + j] * out[ato + 32 * s + 8 * g + j];
    d = rows4(d, [](float a, float b) { return a + b; });
  } else {
    __shared__ float total[C::NG * 16 * C::NW];
    walk<0>(
        nb, [&](int i) { vb.load(v, ld, i * C::BLK, S, tid); },
        [&]() {
          load_p(next++);
          vb.store(vl, tid);
        },
        [&](int) {
          float part = 0.0f;
#pragma unroll
          for (int n = 0; n < N16; n += 2) {
            f4 dp[2];
            blocks32<C>(dp, vl, n0 + n, own, c, g);
#pragma unroll
            for (int u = 0; u < 2; ++u)
#pragma unroll
              for (int e = 0; e < 4; ++e) part += p[n + u][e] * dp[u][e];
          }
          d += part;
        });
    d = rows4(d, [](float a, float b) { return a + b; }) * kUnscale;
    const int r = wave % C::NW * 16 + c;
    if (g == 0) total[grp * 16 * C::NW + r] = d;
    __syncthreads();
    d = total[r];
#pragma unroll
    for (int n = 1; n < C::NG; ++n) d += total[n * 16 * C::NW + r];
    if (__any(live && !(d * 0.0f == 0.0f))) {  // not finite: again in fp32
      using F = Fp32<C>;
      F f;
      f.set(dout + ato, dh, g);
      d = 0.0f;
      for (int r0 = 0; r0 < S; r0 += F::ROWS) {
        typename F::Rows vr;
        vr.load(v, ld, r0, S, dh, c, g);
        f4 dp[F::N];
        f.dots(dp, vr);
#pragma unroll
        for (int u = 0; u < F::N; ++u) {
          const f4 q = load4(Pr, r0 + 16 * u + 4 * g, S, false);
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (r0 + 16 * u + 4 * g + e < S) d += q[e] * dp[u][e];
        }
      }
      d = rows4(d, [](float a, float b) { return a + b; });
    }
    next = 0;
  }
  if (MODE != kGivenD && D != nullptr && live && g == 0 && grp == 0) D[(int64_t)z * S + row] = d;
  if (dq == nullptr) return;
  walk<0>(
      nb,
      [&](int i) {
        vb.load(v, ld, i * C::BLK, S, tid);
        kb.load(k, ld, i * C::BLK, S, tid);
      },
      [&]() {
        load_p(next++);
        vb.store(vl, tid);
        kb.store(kl, tid);
      },
      [&](int i) {
#pragma unroll
        for (int n = 0; n < N16; n += 2) {
          const float sign = (i * (C::SUB / 32) + n / 2) & 1 ? -1.0f : 1.0f;
          float ds[8];
          f4 dp[2];
          blocks32<C>(dp, vl, n0 + n, own, c, g);
#pragma unroll
          for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int e = 0; e < 4; ++e)
              ds[4 * u + e] = sign * kScale * (p[n + u][e] * __builtin_fmaf(dp[u][e], kUnscale, -d));
          Terms t;
          t.set(ds);
          rows32<C>(acc, kl, (n0 + n) / 2, t, sign, c, g);
        }
      });
  join_groups<C>(acc, lds, wave, lane);
  if (grp > 0) return;
  if (any_bad(acc, live)) {
#pragma unroll
    for (int b = 0; b < C::NB; ++b) acc[b] = f4{};
    using F = Fp32<C>;
    F f;
    f.set(dout + ato, dh, g);
    for (int r0 = 0; r0 < S; r0 += F::ROWS) {
      typename F::Rows vr;
      typename F::Cols kr;
      vr.load(v, ld, r0, S, dh, c, g);
      kr.load(k, ld, r0, S, dh, c, g);
      f4 dp[F::N], ds[F::N];
      f.dots(dp, vr);
#pragma unroll
      for (int u = 0; u < F::N; ++u) {
        const int at = r0 + 16 * u + 4 * g;
        const f4 p = load4(Pr, at, S, false);
#pragma unroll
        for (int e = 0; e < 4; ++e) ds[u][e] = at + e < S ? p[e] * (dp[u][e] - d) : 0.0f;
      }
      F::add(acc, kr, ds);
    }
  }
  if (live) store_rows<C>(dq + at + (int64_t)row * ld, acc, alpha, dh, g, add);
}

// dV and dK (either may be null), given D (of head z).  Workgroup blk of head z; lds: three images.
template <class C>
__device__ __forceinline__ void bwd_key(char *lds, int z, int blk, const float *q, const float *v, int ld,
                                        const float *P, const float *dout, int ldo, const float *D, float *dk,
                                        float *dv, int S, int H, int dh, float alpha, int add) {
  static_assert(C::parts_fit(3), "partial outputs");
  char *const ol = lds, *const otl = lds + C::kImage, *const ql = lds + 2 * C::kImage;
  constexpr int N16 = C::N16;
  const int tid = threadIdx.x, lane = tid & 63, c = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), grp = wave / C::NW, n0 = grp * N16;
  const int row = blk * 16 * C::NW + wave % C::NW * 16 + c;
  const bool live = row < S;
  const int rc = min(row, S - 1);
  const int64_t at = (int64_t)(z / H) * S * ld + (z % H) * dh;
  const float *vr = v + at + (int64_t)rc * ld;
  q += at;
  dout += (int64_t)(z / H) * S * ldo + (z % H) * dh;
  Terms own[C::NS];
  own_rows<C>(own, vr, dh, g);
  const float *Pc = P + (int64_t)z * S * S + rc;
  Block<C, false> ob;
  Block<C, true> otb, qb;
  const int nb = (S + C::BLK - 1) / C::BLK;
  f4 av[C::NB], ak[C::NB];
#pragma unroll
  for (int b = 0; b < C::NB; ++b) av[b] = ak[b] = f4{};
  auto load_p = [&](int r0, bool whole) {
    f4 p = {};
    const float *pr = Pc + (int64_t)r0 * S;
    if (whole) {
#pragma unroll
      for (int e = 0; e < 4; ++e) p[e] = pr[e * S];
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (r0 + e < S) p[e] = pr[e * S];
    }
    return p;
  };
  ob.init(ldo, dh, tid);
  otb.init(ldo, dh, tid);
  qb.init(ld, dh, tid);
  auto first = [&](int i) { return i * C::BLK + grp * C::SUB; };
  f4 p[N16], d[N16];
  int next = 0;
  walk<0>(
      nb,
      [&](int i) {
        ob.load(dout, ldo, i * C::BLK, S, tid);
        otb.load(dout, ldo, i * C::BLK, S, tid);
        qb.load(q, ld, i * C::BLK, S, tid);
      },
      [&]() {
        const int r0 = first(next++);
        const bool whole = r0 + C::SUB <= S;
#pragma unroll
        for (int n = 0; n < N16; ++n) {
          p[n] = load_p(r0 + 16 * n + 4 * g, whole);
          d[n] = load4(D, r0 + 16 * n + 4 * g, S, whole);
        }
        ob.store(ol, tid);
        otb.store(otl, tid);
        qb.store(ql, tid);
      },
      [&](int i) {
#pragma unroll
        for (int n = 0; n < N16; n += 2) {
          const float sign = (i * (C::SUB / 32) + n / 2) & 1 ? -1.0f : 1.0f;
          float pv[8], ds[8];
          f4 dp[2];
          blocks32<C>(dp, ol, n0 + n, own, c, g);
#pragma unroll
          for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              pv[4 * u + e] = sign * kScale * p[n + u][e];
              ds[4 * u + e] = sign * kScale * (p[n + u][e] * __builtin_fmaf(dp[u][e], kUnscale, -d[n + u][e]));
            }
          Terms t;
          t.set(pv);
          rows32<C>(av, otl, (n0 + n) / 2, t, sign, c, g);
          t.set(ds);
          rows32<C>(ak, ql, (n0 + n) / 2, t, sign, c, g);
        }
      });
  join_groups<C>(av, lds, wave, lane);
  join_groups<C>(ak, lds, wave, lane);
  if (grp > 0) return;
  if (any_bad(av, live) || any_bad(ak, live)) {
#pragma unroll
    for (int b = 0; b < C::NB; ++b) av[b] = ak[b] = f4{};
    using F = Fp32<C>;
    F f;
    f.set(vr, dh, g);
    for (int r0 = 0; r0 < S; r0 += F::ROWS) {
      typename F::Rows rows;
      typename F::Cols ocols, qcols;
      rows.load(dout, ldo, r0, S, dh, c, g);
      ocols.load(dout, ldo, r0, S, dh, c, g);
      qcols.load(q, ld, r0, S, dh, c, g);
      f4 dp[F::N], p[F::N], ds[F::N];
      f.dots(dp, rows);
#pragma unroll
      for (int u = 0; u < F::N; ++u) {
        const int at = r0 + 16 * u + 4 * g;
        p[u] = load_p(at, false);
        const f4 d = load4(D, at, S, false);
#pragma unroll
        for (int e = 0; e < 4; ++e) ds[u][e] = at + e < S ? p[u][e] * (dp[u][e] - d[e]) : 0.0f;
      }
      F::add(av, ocols, p);
      F::add(ak, qcols, ds);
    }
  }
  if (live) {
    if (dv != nullptr) store_rows<C>(dv + at + (int64_t)row * ld, av, 1.0f, dh, g, add);
    if (dk != nullptr) store_rows<C>(dk + at + (int64_t)row * ld, ak, alpha, dh, g, add);
  }
}

template <class C, int MODE>
__global__ void __launch_bounds__(C::NT) bwd_query_kernel(const float *k, const float *v, int ld, const float *P,
                                                          const float *dout, const float *out, int64_t ldo,
                                                          float *D, float *dq, int S, int H, int dh, float alpha,
                                                          int add) {
  __shared__ __attribute__((aligned(1024))) char lds[2 * C::kImage];
  int z, blk;
  place(z, blk);
  bwd_query<C, MODE>(lds, z, blk, k, v, ld, P, dout, out, ldo, D, dq, S, H, dh, alpha, add);
}

template <class C>
__global__ void __launch_bounds__(C::NT) bwd_key_kernel(const float *q, const float *v, int ld, const float *P,
                                                        const float *dout, int ldo, const float *D, float *dk,
                                                        float *dv, int S, int H, int dh, float alpha, int add) {
  __shared__ __attribute__((aligned(1024))) char lds[3 * C::kImage];
  int z, blk;
  place(z, blk);
  bwd_key<C>(lds, z, blk, q, v, ld, P, dout, ldo, D + (int64_t)z * S, dk, dv, S, H, dh, alpha, add);
}

// Both at once, for heads of at most 64 and S <= kMaxS: 2 x nx workgroups a head.  With the
// forward's output the key ones form the head's D = dO . O themselves; else D is given.  A
// workgroup's chain of loads, splits and MFMAs bounds either kind, so that where one launch leaves
// CUs idle the two together take little longer than one: with the output 64 x 128 x 64 (heads x S x
// dh) 20 -> 12 us, 16 x 256 x 64 30 -> 18, 8 x 512 x 64 49 -> 30; without, D's own launch
// included, 64 x 128 x 64
// 21 -> 17, 32 x 256 x 64 33 -> 25, 16 x 512 x 64 56 -> 41.
constexpr int kMaxS = 512;
template <class C, bool OUT>
__global__ void __launch_bounds__(C::NT) bwd_both_kernel(const float *q, const float *k, const float *v, int ld,
                                                         const float *P, const float *dout, const float *out,
                                                         int ldo, float *D, float *dq, float *dk, float *dv, int S,
                                                         int H, int dh, float alpha, int add) {
  static_assert(C::DH <= 64 && C::NT % 8 == 0, "eight lanes a row");
  __shared__ __attribute__((aligned(1024))) char lds[3 * C::kImage];
  int z, blk;
  place(z, blk);
  const int nx = gridDim.x / 2;
  if (blk < nx) {
    bwd_query<C, OUT ? kOutD : kGivenD>(lds, z, blk, k, v, ld, P, dout, out, ldo, OUT ? nullptr : D, dq, S, H, dh,
                                        alpha, add);
  } else if constexpr (!OUT) {
    bwd_key<C>(lds, z, blk - nx, q, v, ld, P, dout, ldo, D + (int64_t)z * S, dk, dv, S, H, dh, alpha, add);
  } else {
    __shared__ __attribute__((aligned(16))) float Dz[kMaxS];
    const int64_t at = (int64_t)(z / H) * S * ldo + (z % H) * dh;
    const int col = threadIdx.x % 8 * 8;
#pragma unroll 2
    for (int r0 = 0; r0 < S; r0 += C::NT / 8) {
      const int r = r0 + threadIdx.x / 8;
      const int64_t from = at + (int64_t)min(r, S - 1) * ldo + (col < dh ? col : 0);
      float d = 0.0f;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const f4u a = *reinterpret_cast<const f4u *>(dout + from + 4 * h);
        const f4u b = *reinterpret_cast<const f4u *>(out + from + 4 * h);
#pragma unroll
        for (int j = 0; j < 4; ++j) d += a[j] * b[j];
      }
      if (col >= dh) d = 0.0f;
#pragma unroll
      for (int m = 1; m < 8; m *= 2) d += __shfl_xor(d, m);
      if (r < S && col == 0) Dz[r] = d;
    }
    // the first barrier of bwd_key's walk stands before any read of Dz
    bwd_key<C>(lds, z, blk - nx, q, v, ld, P, dout, ldo, Dz, dk, dv, S, H, dh, alpha, add);
  }
}

}  // namespace attn
