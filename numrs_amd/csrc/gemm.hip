// GEMMs for matmul_backward (dA = dC @ B^T, dB = A^T @ dC) and the forward
// products, on gfx950 (CDNA4).
//
// Every product is C[P,Q] (+)= X[P,R] @ Y[R,Q] where each operand is either
// "R-contiguous" (the reduction index is the fast one in memory: X[p*ld + r],
// Y[q*ld + r]) or "P/Q-contiguous" (X[r*ld + p], Y[r*ld + q]).  The four
// layouts cover every product on the path:
//   dA = dC @ B^T   X = dC (R-contig), Y = B   (R-contig)   [NT]
//   dB = A^T @ dC   X = A  (P-contig), Y = dC  (Q-contig)   [TN]
//   C  = A @ B      X = A  (R-contig), Y = B   (Q-contig)   [NN]
//   y  = x @ W^T    X = x  (R-contig), Y = W   (R-contig)   [NT]
//
// Work decomposition
//   * Tiny products (a small batch's layers): 16 x 16 blocks, fp32 MFMAs, one
//     launch (tiny_gemm_kernel).
//   * All others: output tiles of four sizes (kShapes), the products formed on
//     the bf16 matrix cores from three-term splits of the fp32 operands
//     (gemm_bf3.h), any sizes, strides and alignment.  plan_product picks the
//     tile and the split-K ranges per product.
//   * A gradient pair (matmul_backward's dA and dB, a Linear's dx and dW)
//     launches both products' tiles in one grid.
//   * XCD-aware ordering: gfx950 dispatches workgroup b to XCD b % 8; the
//     logical tile index is permuted so each XCD owns a contiguous run of
//     tiles and its private L2 sees the operand rows/columns it reuses.
//   * Split-K for products with few output tiles and long reductions (the
//     weight gradients X^T dY of Linear layers): each split writes a plain
//     partial, splitk_reduce adds them in split order -- deterministic.
#include <algorithm>
#include <type_traits>

#include "common.h"
#include "gemm_bf3.h"

namespace {

typedef float f4 __attribute__((ext_vector_type(4)));

using bf3::kBR;
constexpr int kGroupRows = 4;            // tile rows per raster group

struct Gemm {
  const float *X;
  const float *Y;
  float *C;
  int64_t ldx, ldy, ldc;
  // Batch z = zo * binner + zi addresses X + zo*bsx + zi*bsx2 (same for Y, C):
  // one level covers plain batches, two levels cover head-interleaved
  // layouts such as [batch, seq, heads, dim].
  int64_t bsx, bsy, bsc;
  int64_t bsx2, bsy2, bsc2;
  int binner;
  int P, Q, R;
  int tiles_p, tiles_q;
  int accumulate;
  float alpha;  // C = alpha * X@Y (+ C)
  // Split-K: with splits > 1 the reduction is cut into `splits` ranges of
  // whole k-tiles; range s of batch z writes its plain partial product to
  // partial + (z*splits + s)*P*Q (row stride Q) and splitk_reduce forms
  // alpha*sum (+C).
  int splits;
  int ktiles_per_split;
  float *partial;
  // Optional bias added per output column after alpha: C = alpha*X@Y + bias[q]
  // (+ C); the Linear forward's "+ b" folded into the product's epilogue.
  const float *bias;
  // Tiny kernel only: X entries whose `xmask` entry (same layout and
  // offsets as X) is not > 0 read as zero (ReLU backward applied on load).
  const float *xmask;
  // Activation applied last in the epilogue (batch-1 products): kActRelu
  // (x.max(0)) or kActGelu (exact erf); with `pre` the value before it is
  // stored there too (row stride ldc), for the activation's backward.
  int act;
  float *pre;
  // Optional residual added after the bias: C = alpha*X@Y + bias[q] +
  // res[p*ldr + q] (+ C) -- the "x + Linear(a)" of a residual block folded
  // into the product's epilogue (batch-1 products).
  const float *res;
  int64_t ldr;
  // Tiny kernel only: split products reduced inside their own launch have one
  // arrival counter per output block; null otherwise.
  unsigned *arrive;
  // gemm_pair_kernel<..., SUMS>, the second product: sums[p] (+)= sum_r X[p, r]; split, the
  // partial sums of range s at sums + s*P.
  float *sums;
  int sums_acc;
};

// Epilogue activations: the ReLU forward kernel's x.max(0) and the unary
// kernel's exact-erf GELU, value for value.
constexpr int kActRelu = 1, kActGelu = 2;
__device__ __forceinline__ float act_value(int act, float v) {
  return act == kActRelu ? fmaxf(v, 0.0f) : numrs_hip::gelu_erf(v);
}

// One split product's reduction: C = alpha * sum_s partial[s] (+ bias[q])
// (+ C), partial s at partial + s*n with row stride Q; batch z (blockIdx.z) at
// partial + z*splits*n, its C as Gemm's.
struct SplitSet {
  const float *partial;
  float *C;
  const float *bias;
  int64_t ldc, n;
  int Q, splits, acc;
  float alpha;
  int act;     // activation applied last (Gemm::act)
  float *pre;  // optional pre-activation output (row stride ldc)
  const float *res;  // residual added after the bias (row stride ldr)
  int64_t ldr;
  int kahan;  // the splits added as a compensated (Kahan) sum, in the same order
  int64_t bsc, bsc2;
  int binner;
};

// Column sums out[c] (+)= sum_r g[r ldg + c] of a [rows, cols] block in one
// pass, carried by the launch that reduces a product's splits or on their own
// (a bias gradient where its Linear has no dx or no dW, or an LSTM layer's).  A workgroup owns eight columns
// (two float4 groups; cols % 4 == 0, a last group past the end is skipped)
// and 128 row classes: thread k reads chunk k % 2 of rows k / 2, k / 2 + 128,
// ... and adds them in order, 16 loads in flight; the 128 class sums of a
// column are then added through LDS in a fixed order (32 sums of four
// consecutive classes, then those 32 in order) -- deterministic.  Two lanes
// read 32 contiguous bytes of a row (four columns per workgroup, one lane
// per row, measured 12.3 against 9.6 us for [4096, 1536]).  Consecutive
// column groups run on one XCD, so the workgroups that share a cache line
// read it through the same L2.
struct ColSum {
  const float *g;
  float *out;
  int64_t rows, cols, ldg;
  int acc;
  const float *mask;  // tiny kernel only (see tiny_colsum)
};
constexpr int kColSumCols = 8;
constexpr int kColSumLanes = kColSumCols / 4;       // lanes reading one row's columns
constexpr int kColSumClasses = 256 / kColSumLanes;  // row classes of a workgroup

// Column groups of a [., cols] block.
__host__ __device__ inline int64_t colsum_groups(int64_t cols) { return (cols + kColSumCols - 1) / kColSumCols; }

// A workgroup of 256.
__device__ __forceinline__ void colsum_block(const ColSum &c, int64_t blk) {
  __shared__ f4 red[256];
  const int k = threadIdx.x;
  const int j = k % kColSumLanes, rc = k / kColSumLanes;  // column chunk, row class
  const float *p = c.g + blk * kColSumCols + 4 * j;
  const bool live = blk * kColSumCols + 4 * j < c.cols;
  f4 s = {0.0f, 0.0f, 0.0f, 0.0f};
  for (int64_t r0 = rc; live && r0 < c.rows; r0 += kColSumClasses * 16) {
    f4 v[16];
#pragma unroll
    for (int u = 0; u < 16; ++u) {
      const int64_t r = r0 + kColSumClasses * u;
      v[u] = r < c.rows ? *reinterpret_cast<const f4 *>(p + r * c.ldg) : f4{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int u = 0; u < 16; ++u) s += v[u];
  }
  red[k] = s;  // k = kColSumLanes * class + chunk
  __syncthreads();
  // 64 partials: chunk t % lanes, classes 4 (t / lanes) .. + 3, added in order
  f4 t = {0.0f, 0.0f, 0.0f, 0.0f};
  if (k < 64) {
    const int jj = k % kColSumLanes, g = k / kColSumLanes;
    t = ((red[kColSumLanes * (4 * g) + jj] + red[kColSumLanes * (4 * g + 1) + jj]) +
         red[kColSumLanes * (4 * g + 2) + jj]) +
        red[kColSumLanes * (4 * g + 3) + jj];
  }
  __syncthreads();
  if (k < 64) red[k] = t;
  __syncthreads();
  const int64_t gc = blk * kColSumCols + k;
  if (k < kColSumCols && gc < c.cols) {
    const int jj = k / 4, e = k % 4;
    float u = 0.0f;
    for (int g = 0; g < 64 / kColSumLanes; ++g) u += red[kColSumLanes * g + jj][e];
    c.out[gc] = c.acc ? c.out[gc] + u : u;
  }
}

// Workgroup b of a launch row of n workgroups (hardware ids go to the eight
// XCDs in turn, n % 8 == 0) -> column group, so that XCD x owns groups
// [x m/8, (x+1) m/8) of the m groups; -1 for a workgroup with no group.
__device__ __forceinline__ int64_t colsum_group(int b, int n, int64_t m) {
  if ((n & 7) != 0 || (m & 7) != 0) return b < m ? b : -1;
  const int64_t idx = b >> 3;
  return idx < (m >> 3) ? (b & 7) * (m >> 3) + idx : -1;
}

// The end of a split reduction at C[p, q] made inside a product's launch (tiny_tile): alpha, bias,
// residual, accumulate, activation (pre-activation stored first), as splitk_reduce's epilogue,
// operation for operation.
__device__ __forceinline__ void finish_split(float *C, const Gemm &d, int64_t p, int64_t q, float s) {
  float *dst = C + p * d.ldc + q;
  float v = d.alpha * s;
  if (d.bias != nullptr) v = v + d.bias[q];
  if (d.res != nullptr) v = v + d.res[p * d.ldr + q];
  v = d.accumulate ? *dst + v : v;
  if (d.act) {
    if (d.pre != nullptr) d.pre[p * d.ldc + q] = v;
    v = act_value(d.act, v);
  }
  *dst = v;
}

// Splits are added in order s = 0, 1, ... (deterministic); the loads of a
// batch of splits are issued before its ordered adds.  With column sums
// (has_cs), row y = 0 of the grid computes them and rows 1, 2, 3 reduce the
// sets; otherwise rows 0, 1, 2 reduce the sets.  The column sums (one
// long strided walk per workgroup) go first so that they are dispatched
// before, and overlap, the short split reductions.  VEC: four consecutive
// elements of one row per thread (Q, ldc and the pointers 16-byte aligned).
template <bool VEC>
__global__ void __launch_bounds__(256) splitk_reduce(SplitSet s0, SplitSet s1, SplitSet s2,
                                                     ColSum cs, int has_cs) {
  if (has_cs && blockIdx.y == 0) {
    const int64_t grp = colsum_group(blockIdx.x, gridDim.x, colsum_groups(cs.cols));
    if (grp >= 0) colsum_block(cs, grp);
    return;
  }
  const int y = (int)blockIdx.y - has_cs;
  const SplitSet &d = y == 0 ? s0 : y == 1 ? s1 : s2;
  int64_t from = 0, to = 0;  // batch z's partials and C
  if (gridDim.z > 1) {
    const unsigned z = blockIdx.z, zo = z / (unsigned)d.binner, zi = z - zo * (unsigned)d.binner;
    from = (int64_t)z * d.splits * d.n;
    to = zo * d.bsc + zi * d.bsc2;
  }
  typedef typename std::conditional<VEC, f4, float>::type V;
  constexpr int kW = VEC ? 4 : 1;
  constexpr int kBatch = VEC ? 4 : 8;
  const int64_t e = ((int64_t)blockIdx.x * 256 + threadIdx.x) * kW;
  if (e >= d.n) return;
  V s = V{}, comp = V{};
  for (int k0 = 0; k0 < d.splits; k0 += kBatch) {
    V v[kBatch];
#pragma unroll
    for (int u = 0; u < kBatch; ++u)
      if (k0 + u < d.splits) v[u] = *reinterpret_cast<const V *>(d.partial + from + (k0 + u) * d.n + e);
    if (d.kahan) {
#pragma unroll
      for (int u = 0; u < kBatch; ++u)
        if (k0 + u < d.splits) {
          const V y = v[u] - comp;
          const V t = s + y;
          comp = (t - s) - y;
          s = t;
        }
    } else {
#pragma unroll
      for (int u = 0; u < kBatch; ++u)
        if (k0 + u < d.splits) s += v[u];
    }
  }
  const int64_t p = e / d.Q, q = e - p * d.Q;
  V *dst = reinterpret_cast<V *>(d.C + to + p * d.ldc + q);
  V v = d.alpha * s;
  if (d.bias != nullptr) v = v + *reinterpret_cast<const V *>(d.bias + q);
  if (d.res != nullptr) v = v + *reinterpret_cast<const V *>(d.res + p * d.ldr + q);
  v = d.acc ? *dst + v : v;
  if (d.act) {
    if (d.pre != nullptr) *reinterpret_cast<V *>(d.pre + p * d.ldc + q) = v;
    if constexpr (VEC) {
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = act_value(d.act, v[e]);
    } else {
      v = act_value(d.act, v);
    }
  }
  *dst = v;
}

// Output tile (tp, tq) of logical tile `tile`: tiles run in groups of
// kGroupRows tile rows, column by column within a group.
__device__ __forceinline__ void tile_rc(int tiles_p, int tiles_q, int tile, int &tp, int &tq) {
  const int per_group = kGroupRows * tiles_q;
  const int gidx = tile / per_group;
  const int first_p = gidx * kGroupRows;
  const int rows_in_group = min(tiles_p - first_p, kGroupRows);
  const int in_group = tile - gidx * per_group;
  tp = first_p + in_group % rows_in_group;
  tq = in_group / rows_in_group;
}

// Maps the hardware workgroup (x fastest, XCD = linear id % 8) to a logical
// (tile, batch) so that each XCD owns a contiguous run of the batch-major
// logical ids, whose tiles share operand panels through its L2.
__device__ __forceinline__ void xcd_tile(int &tile, int &batch) {
  const int nx = gridDim.x, nb = nx * gridDim.y, lin = blockIdx.x + nx * blockIdx.y;
  const int xcd = lin & 7, per = nb >> 3, more = nb & 7;
  const int logical = xcd * per + min(xcd, more) + (lin >> 3);
  batch = logical / nx;
  tile = logical - batch * nx;
}

// Workgroup tiles, largest first.  L: eight waves of 64 x 64 outputs, 144 KiB
// of LDS, one per CU.  M: eight waves of 64 x 32, 96 KiB, one per CU.  N: four
// waves of 64 x 32, 72 KiB, two per CU.  S: four waves of 32 x 32, 48 KiB,
// three per CU; also takes leading dimensions of 2^24 and more.
using ShapeL = bf3::Shape<4, 4, 4, 2, false>;
using ShapeM = bf3::Shape<4, 2, 2, 4, false>;
using ShapeN = bf3::Shape<4, 2, 2, 2, false>;
using ShapeS = bf3::Shape<2, 2, 2, 2, true>;
template <class S>
constexpr int kWavesPerSimd = std::is_same<S, ShapeS>::value ? 3 : 2;

// ACT: the epilogue applies d.act (and stores d.pre); a separate
// instantiation, so products without an activation keep the plain epilogue.
// Splits are the slow index of the logical tiles: the tiles that an XCD runs
// at a time are mostly of one reduction range and share its operand panels.
// SUMS: tiles of the first tile column also form d.sums, the sums of X's rows, from the values
// that the loader holds (four threads a row, each the sum over tiles of eight steps): a Linear's
// bias gradient without another pass over its output gradient.  In an encoder block's step (4096
// tokens) the split reductions that read it took 12.3 + 14.4 + 9.6 + 14.0 us and take 5.1 +
// 10.2 + 4.8 + 7.7, the 128 x 128 pairs 112 -> 116 and 32 -> 35 us, the 256 x 128 ones what
// they did; 1001 x 777 -> 1531 forward and backward 96 -> 86 us (it had two more launches).
template <bool XRC, bool YRC, class S, bool ACT = false, bool SUMS = false>
__device__ __forceinline__ void bf3_tile(const Gemm &d, int tile, int batch, char *lds) {
  constexpr int BI = S::BI, BJ = S::BJ;
  const int n = d.tiles_p * d.tiles_q;
  const int split = tile / n;
  int tp, tq;
  tile_rc(d.tiles_p, d.tiles_q, tile - split * n, tp, tq);
  const int p0 = tp * S::TP, q0 = tq * S::TQ;
  const int64_t r0 = (int64_t)split * d.ktiles_per_split * kBR;
  const int R = (int)min(d.R - r0, (int64_t)d.ktiles_per_split * kBR);
  const int64_t zo = batch / d.binner, zi = batch - zo * d.binner;
  const float *X = d.X + zo * d.bsx + zi * d.bsx2 + (XRC ? p0 * d.ldx + r0 : p0 + r0 * d.ldx);
  const float *Y = d.Y + zo * d.bsy + zi * d.bsy2 + (YRC ? q0 * d.ldy + r0 : q0 + r0 * d.ldy);
  bf3::Product<XRC, YRC, S, SUMS> prod;
  prod.run(X, d.ldx, min(S::TP, d.P - p0), Y, d.ldy, min(S::TQ, d.Q - q0), R,
           tp ^ tq ^ split ^ batch, lds);
  if constexpr (SUMS) {
    if (tq == 0) {
      using L = typename bf3::Product<XRC, YRC, S, SUMS>::LX;
      float *const red = reinterpret_cast<float *>(lds);  // [chunk][row]
      const int tid = threadIdx.x, rows = min(S::TP, d.P - p0);
      __syncthreads();
#pragma unroll
      for (int i = 0; i < L::N; ++i)
        red[L::chunk(tid, i) * S::TP + L::read_row(tid, i, rows)] = prod.rowsum[i];
      __syncthreads();
      if (tid < rows) {
        const float v = (red[tid] + red[S::TP + tid]) + (red[2 * S::TP + tid] + red[3 * S::TP + tid]);
        float *out = d.sums + (d.splits > 1 ? (int64_t)split * d.P : 0) + p0 + tid;
        *out = d.sums_acc ? *out + v : v;
      }
    }
  }

  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int pl = p0 + (wave / S::WQ) * (16 * BI) + 4 * (lane >> 4);  // + 16 i + e
  const int ql = q0 + (wave % S::WQ) * (16 * BJ) + (lane & 15);      // + 16 j
  // FULL: a tile wholly inside the output, no guards.
  auto finish = [&](auto full_t) {
    constexpr bool FULL = decltype(full_t)::value;
    auto in = [&](int i, int j, int e) {
      return FULL || (pl + 16 * i + e < d.P && ql + 16 * j < d.Q);
    };
    if (d.splits > 1) {  // plain partial product, row stride Q; splitk_reduce finishes
      float *part = d.partial + ((int64_t)batch * d.splits + split) * d.P * d.Q;
#pragma unroll
      for (int i = 0; i < BI; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int j = 0; j < BJ; ++j)
            if (in(i, j, e)) part[(int64_t)(pl + 16 * i + e) * d.Q + ql + 16 * j] = prod.tot[i][j][e];
      return;
    }
    // Residual and bias values are all loaded before the first store: res may
    // alias C, which would otherwise order each load after the previous store.
    float bq[BJ];
#pragma unroll
    for (int j = 0; j < BJ; ++j)
      bq[j] = d.bias != nullptr && (FULL || ql + 16 * j < d.Q) ? d.bias[ql + 16 * j] : 0.0f;
    f4 rv[BI][BJ];
    if (d.res != nullptr) {
#pragma unroll
      for (int i = 0; i < BI; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int j = 0; j < BJ; ++j)
            rv[i][j][e] = in(i, j, e) ? d.res[(int64_t)(pl + 16 * i + e) * d.ldr + ql + 16 * j] : 0.0f;
    }
    float *C = d.C + zo * d.bsc + zi * d.bsc2;
#pragma unroll
    for (int i = 0; i < BI; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int j = 0; j < BJ; ++j)
          if (in(i, j, e)) {
            const int64_t at = (int64_t)(pl + 16 * i + e) * d.ldc + ql + 16 * j;
            float v = d.alpha * prod.tot[i][j][e];
            if (d.bias != nullptr) v = v + bq[j];
            if (d.res != nullptr) v = v + rv[i][j][e];
            v = d.accumulate ? C[at] + v : v;
            if constexpr (ACT) {
              if (d.pre != nullptr) d.pre[at] = v;
              v = act_value(d.act, v);
            }
            C[at] = v;
          }
  };
  if (p0 + S::TP <= d.P && q0 + S::TQ <= d.Q)
    finish(std::true_type{});
  else
    finish(std::false_type{});
}

template <bool XRC, bool YRC, class S, bool ACT = false>
__global__ void __launch_bounds__(S::NT, kWavesPerSimd<S>) gemm_kernel(Gemm d) {
  __shared__ __attribute__((aligned(1024))) char lds[S::kLds];
  int tile, batch;
  xcd_tile(tile, batch);
  bf3_tile<XRC, YRC, S, ACT>(d, tile, batch, lds);
}

// Two products in one grid: logical tiles [0, tiles_a) belong to `a`, the
// rest to `b`, which is TN.  matmul_backward: dA = dC B^T (NT) with dB =
// A^T dC; the Linear backward: dx = g W (NN) with dW = g^T x; two weight
// gradients (TN).
template <bool XA, bool YA, class S, bool SUMS = false>
__global__ void __launch_bounds__(S::NT, kWavesPerSimd<S>) gemm_pair_kernel(Gemm a, Gemm b,
                                                                            int tiles_a) {
  __shared__ __attribute__((aligned(1024))) char lds[S::kLds];
  int tile, batch;
  xcd_tile(tile, batch);
  if (tile < tiles_a)
    bf3_tile<XA, YA, S>(a, tile, batch, lds);
  else
    bf3_tile<false, false, S, false, SUMS>(b, tile - tiles_a, batch, lds);
}

void apply_splits(Gemm &g, int splits, float *partial) {
  const int nk = (g.R + kBR - 1) / kBR;
  g.splits = splits;
  g.ktiles_per_split = (nk + splits - 1) / splits;
  g.partial = partial;
}

// Whether the column sums of g [rows, cols] (row stride ldg) can ride in the
// split-reduce launch: float4 column groups and at most 8192 rows (a
// workgroup walks every row of its eight columns).
bool colsum_fits(const float *g, int64_t rows, int64_t cols, int64_t ldg) {
  return cols % 4 == 0 && ldg % 4 == 0 && numrs_hip::aligned16(g) && rows <= 8192 &&
         cols / kColSumCols <= 0x7ffffff0;
}

// Reduces the split products among a and b (either may be null or unsplit)
// with one launch, which also forms the column sums `cs` when given and
// reduces the set `extra` (then the launch is made even when nothing was
// split).
int reduce_splits(numrs_hip_ctx *ctx, const Gemm *a, const Gemm *b, const ColSum *cs = nullptr,
                  const SplitSet *extra = nullptr, int64_t batch = 1) {
  const Gemm *g[2];
  int m = 0;
  if (a != nullptr && a->splits > 1) g[m++] = a;
  if (b != nullptr && b->splits > 1) g[m++] = b;
  if (m == 0 && cs == nullptr && extra == nullptr) return NUMRS_HIP_OK;
  SplitSet set[3] = {};
  bool vec = true;
  int64_t most = 0;
  for (int i = 0; i < m; ++i) {
    const Gemm &d = *g[i];
    set[i] = SplitSet{d.partial, d.C, d.bias, d.ldc, (int64_t)d.P * d.Q, d.Q, d.splits,
                      d.accumulate, d.alpha, d.act, d.pre, d.res, d.ldr, 0, d.bsc, d.bsc2, d.binner};
  }
  if (extra != nullptr) set[m++] = *extra;
  for (int i = 0; i < m; ++i) {
    const SplitSet &d = set[i];
    vec = vec && d.Q % 4 == 0 && d.ldc % 4 == 0 && d.bsc % 4 == 0 && d.bsc2 % 4 == 0 && numrs_hip::aligned16(d.C) &&
          numrs_hip::aligned16(d.partial) && (d.bias == nullptr || numrs_hip::aligned16(d.bias)) &&
          (d.res == nullptr || (numrs_hip::aligned16(d.res) && d.ldr % 4 == 0)) &&
          (d.pre == nullptr || numrs_hip::aligned16(d.pre));
    most = std::max(most, d.n);
  }
  for (int i = m; i < 3; ++i) set[i] = set[0];
  int64_t blocks = (most / (vec ? 4 : 1) + 255) / 256;
  ColSum c{};
  const int has_cs = cs != nullptr ? 1 : 0;
  if (cs != nullptr) {
    c = *cs;
    blocks = std::max<int64_t>(blocks, colsum_groups(c.cols));
    blocks = (blocks + 7) & ~int64_t{7};  // whole rounds of the eight XCDs
  }
  if (blocks > 0x7fffffff)
    return numrs_hip::fail(ctx, NUMRS_HIP_E_INVALID, "splitk_reduce: too large");
  dim3 grid((unsigned)std::max<int64_t>(blocks, 1), (unsigned)(m + has_cs), (unsigned)batch);
  if (vec)
    splitk_reduce<true><<<grid, 256, 0, ctx->stream>>>(set[0], set[1], set[2], c, has_cs);
  else
    splitk_reduce<false><<<grid, 256, 0, ctx->stream>>>(set[0], set[1], set[2], c, has_cs);
  return numrs_hip::check_launch(ctx, "splitk_reduce");
}

// ---------------------------------------------------------------------------
// Tiny products (a small batch's MLP layers: [64,784] x [784,128],
// [64,128] x [128,10] and their gradients).  128 x 128 tiles would leave all
// but a few CUs idle and walk the reduction serially, so a workgroup owns one
// 16 x 16 output block and its eight waves split the reduction: wave w takes
// the 16-wide reduction steps w, w + 8, ..., four v_mfma_f32_16x16x4f32 per
// step, with operands loaded straight from global memory (L2 serves the reuse
// across blocks); the eight partial blocks are then added in wave order
// through LDS -- deterministic.  One launch carries up to two products (a
// gradient pair) and the column sums of a bias gradient.
//   MFMA 16x16x4 lane contract (lane l = 16 g + i): A row i at reduction slot
//   g; B reduction slot g at column i; D column i, rows 4g + v (v = 0..3).
//   Reduction index k = 16 s + 4 g + j feeds MFMA j of step s at slot g, for
//   A and B alike.
constexpr int kTinyWaves = 8;
constexpr int kTinyThreads = 64 * kTinyWaves;
// Reduction steps per load batch and wave: 8 (143 VGPRs, one workgroup per
// CU) for reductions over 512, else 4 (79 VGPRs, three per CU).
constexpr int kTinyUBig = 8, kTinyUSmall = 4;
constexpr int kTinyColsumCols = 64;
constexpr int kTinyColsumRows = 8192;
constexpr int64_t kTinyMacs = int64_t{1} << 24;
constexpr int kTinyMaxR = 4096;  // at most four load batches per wave

// FUSE (batch 1, d.arrive set for a split product): a split stores its
// partial at device scope and arrives at its output block's counter; the
// last of the block's splits adds the block's partials in split order with
// splitk_reduce's arithmetic (finish_split) and sets the counter
// back to zero -- no reduce launch, and no workgroup waits for another.
template <bool XRC, bool YRC, int U, bool FUSE = false>
__device__ __forceinline__ void tiny_tile(const Gemm &d, int tile, int batch) {
  // Split-K: consecutive logical blocks are the k-ranges of one output block.
  const int split = tile % d.splits;
  tile /= d.splits;
  const int tq_n = (d.Q + 15) >> 4;
  const int tp = tile / tq_n, tq = tile - tp * tq_n;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int i = lane & 15, g = lane >> 4;
  const int p = tp * 16 + i, q = tq * 16 + i;
  const int64_t zo = batch / d.binner, zi = batch - zo * d.binner;
  const float *__restrict__ X = d.X + zo * d.bsx + zi * d.bsx2;
  const float *__restrict__ Y = d.Y + zo * d.bsy + zi * d.bsy2;
  float *__restrict__ C = d.C + zo * d.bsc + zi * d.bsc2;
  const float *__restrict__ M = d.xmask != nullptr ? d.xmask + zo * d.bsx + zi * d.bsx2 : nullptr;
  const bool pin = p < d.P, qin = q < d.Q;
  // This split's 16-wide reduction steps [s_lo, steps); k-tiles are 32 wide.
  const int s_lo = split * d.ktiles_per_split * 2;
  const int steps = min((d.R + 15) >> 4, s_lo + d.ktiles_per_split * 2);
  // Byte offsets from the (wave-uniform) operand bases fit in 32 bits
  // (tiny_fits), so each load needs one VGPR of address.
  const char *Xc = reinterpret_cast<const char *>(X), *Yc = reinterpret_cast<const char *>(Y);
  const char *Mc = reinterpret_cast<const char *>(M);
  const uint32_t ldx4 = 4u * (uint32_t)d.ldx, ldy4 = 4u * (uint32_t)d.ldy;
  const uint32_t xo = XRC ? (uint32_t)p * ldx4 : 4u * (uint32_t)p;  // reduction index 0
  const uint32_t yo = YRC ? (uint32_t)q * ldy4 : 4u * (uint32_t)q;
  const uint32_t xk = XRC ? 4u : ldx4, yk = YRC ? 4u : ldy4;  // bytes per reduction index
  auto ld = [](const char *base, uint32_t off) {
    return *reinterpret_cast<const float *>(base + off);
  };
  f4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
  for (int s0 = s_lo + w; s0 < steps; s0 += kTinyWaves * U) {
    f4 a[U], b[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int s = s0 + kTinyWaves * u;  // wave-uniform
      if (s < steps) {
        const int k = 16 * s + 4 * g;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const bool kin = k + j < d.R;
          const uint32_t xoff = xo + (uint32_t)(k + j) * xk;
          a[u][j] = pin && kin ? ld(Xc, xoff) : 0.0f;
          if (Mc != nullptr) a[u][j] = pin && kin && ld(Mc, xoff) > 0.0f ? a[u][j] : 0.0f;
          b[u][j] = qin && kin ? ld(Yc, yo + (uint32_t)(k + j) * yk) : 0.0f;
        }
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (s0 + kTinyWaves * u < steps)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[u][j], b[u][j], acc, 0, 0, 0);
  }
  __shared__ float part[kTinyWaves][256];
#pragma unroll
  for (int v = 0; v < 4; ++v) part[w][(4 * g + v) * 16 + i] = acc[v];
  __syncthreads();
  if (threadIdx.x < 256) {
    const int t = threadIdx.x;
    float s = part[0][t];
#pragma unroll
    for (int ww = 1; ww < kTinyWaves; ++ww) s += part[ww][t];
    const int pp = tp * 16 + (t >> 4), qq = tq * 16 + (t & 15);
    if (pp < d.P && qq < d.Q && d.splits > 1) {
      float *dst = d.partial + ((int64_t)split * d.P + pp) * d.Q + qq;
      if constexpr (FUSE)
        numrs_hip::st_dev(dst, s);  // read by the block's last split
      else
        *dst = s;  // splitk_reduce finishes
    } else if (pp < d.P && qq < d.Q) {
      float *dst = C + (int64_t)pp * d.ldc + qq;
      float v = d.alpha * s;
      if (d.bias != nullptr) v = v + d.bias[qq];
      if (d.res != nullptr) v = v + d.res[(int64_t)pp * d.ldr + qq];
      v = d.accumulate ? *dst + v : v;
      if (d.act) {
        if (d.pre != nullptr) d.pre[(int64_t)pp * d.ldc + qq] = v;
        v = act_value(d.act, v);
      }
      *dst = v;
    }
  }
  if constexpr (FUSE) {
    if (d.splits > 1) {
      __shared__ int s_last;
      __builtin_amdgcn_s_waitcnt(0);  // this lane's partial stores acknowledged
      __syncthreads();
      if (threadIdx.x == 0) {
        unsigned *ctr = d.arrive + tile;
        const bool last = __hip_atomic_fetch_add(ctr, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ==
                          (unsigned)(d.splits - 1);
        if (last) __hip_atomic_store(ctr, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        s_last = last ? 1 : 0;
      }
      __syncthreads();
      if (s_last != 0 && threadIdx.x < 256) {
        const int t = threadIdx.x;
        const int pp = tp * 16 + (t >> 4), qq = tq * 16 + (t & 15);
        if (pp < d.P && qq < d.Q) {
          const int64_t n = (int64_t)d.P * d.Q, e = (int64_t)pp * d.Q + qq;
          const __amdgpu_buffer_rsrc_t rs = numrs_hip::dev_rsrc(d.partial, (int64_t)d.splits * n * 4);
          float sum = 0.0f;
          for (int k0 = 0; k0 < d.splits; k0 += 8) {
            float v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u)
              if (k0 + u < d.splits) v[u] = numrs_hip::ld_dev1(rs, (int)(4 * ((k0 + u) * n + e)));
#pragma unroll
            for (int u = 0; u < 8; ++u)
              if (k0 + u < d.splits) sum += v[u];
          }
          finish_split(C, d, pp, qq, sum);
        }
      }
    }
  }
}

// Column sums of a small bias gradient: 64 columns per workgroup, thread
// (class k, column c) adds rows k, k + 8, ... in order, and the eight class
// sums are added in class order.  With `mask` (same layout as g), entries
// whose mask is not > 0 count as zero.
__device__ __forceinline__ void tiny_colsum(const ColSum &c, int blk) {
  __shared__ float red[kTinyWaves][kTinyColsumCols];
  const int cl = threadIdx.x & 63, k = threadIdx.x >> 6;
  const int64_t col = (int64_t)blk * kTinyColsumCols + cl;
  float s = 0.0f;
  if (col < c.cols) {
    if (c.mask != nullptr) {
#pragma unroll 8
      for (int64_t r = k; r < c.rows; r += kTinyWaves) {
        const int64_t idx = r * c.ldg + col;
        s += c.mask[idx] > 0.0f ? c.g[idx] : 0.0f;
      }
    } else {
#pragma unroll 8
      for (int64_t r = k; r < c.rows; r += kTinyWaves) s += c.g[r * c.ldg + col];
    }
  }
  red[k][cl] = s;
  __syncthreads();
  if (threadIdx.x < kTinyColsumCols && col < c.cols) {
    float t = red[0][cl];
#pragma unroll
    for (int kk = 1; kk < kTinyWaves; ++kk) t += red[kk][cl];
    c.out[col] = c.acc ? c.out[col] + t : t;
  }
}

// Workgroups [0, tiles_a) form product a (layout XA, YA), the next tiles_b
// product b (TN), the rest (batch 0 only) the column sums cs.
template <bool XA, bool YA, int U, bool FUSE = false>
__global__ void __launch_bounds__(kTinyThreads) tiny_gemm_kernel(Gemm a, Gemm b, int tiles_a,
                                                                 int tiles_b, ColSum cs) {
  const int t = blockIdx.x;
  if (t < tiles_a)
    tiny_tile<XA, YA, U, FUSE>(a, t, blockIdx.y);
  else if (t < tiles_a + tiles_b)
    tiny_tile<false, false, U, FUSE>(b, t - tiles_a, blockIdx.y);
  else if (blockIdx.y == 0)
    tiny_colsum(cs, t - tiles_a - tiles_b);
}

int64_t tiny_tiles(const Gemm &g) { return (int64_t)((g.P + 15) / 16) * ((g.Q + 15) / 16); }

bool tiny_fits(const Gemm &g, int64_t batch) {
  // Each operand's byte extent under either layout stays below 2^31 (the
  // kernel's 32-bit load offsets).
  auto span = [](int64_t ext, int64_t other, int64_t ld) {
    return 4 * std::max((ext - 1) * ld + other, (other - 1) * ld + ext) < (int64_t{1} << 31);
  };
  return g.splits == 1 && g.R <= kTinyMaxR && (int64_t)g.P * g.Q * g.R * batch <= kTinyMacs &&
         span(g.P, g.R, g.ldx) && span(g.Q, g.R, g.ldy);
}

// Split-K for tiny products with few output blocks and a long reduction
// (the first MLP layer: 32 blocks over 784): blocks x splits fill the CUs,
// each split keeping at least four 32-wide k-tiles (a 16-wide step per
// wave); splitk_reduce then adds the splits in order.  A lone workgroup
// per CU streaming a long reduction is bound by its outstanding loads.
int tiny_split(int64_t cus, int64_t blocks, int R) {
  const int64_t kt = (R + kBR - 1) / kBR;
  int64_t sp = std::min<int64_t>({(cus + blocks - 1) / blocks, kt / 4, 32});
  if (sp <= 1) return 1;
  const int64_t per = (kt + sp - 1) / sp;
  return (int)((kt + per - 1) / per);
}

// One launch of the tiny kernel: product a (layout xa, ya), optionally a TN
// product b, and (batch 1) the column sums cs; then the split reduction
// when a batch-1 product was split.
int launch_tiny(numrs_hip_ctx *ctx, const Gemm &a_in, bool xa, bool ya, const Gemm *b_in,
                int64_t batch, const ColSum *cs) {
  Gemm a = a_in, bb = b_in != nullptr ? *b_in : a_in;
  const Gemm *b = b_in != nullptr ? &bb : nullptr;
  int64_t ta = tiny_tiles(a), tb = b != nullptr ? tiny_tiles(*b) : 0;
  const int64_t tc = cs != nullptr ? (cs->cols + kTinyColsumCols - 1) / kTinyColsumCols : 0;
  if (ta + tb + tc > 0x7fffffff || batch < 1 || batch > 65535 || (cs != nullptr && batch != 1))
    return numrs_hip::fail(ctx, NUMRS_HIP_E_INVALID, "tiny_gemm: bad launch shape");
  int sa = 1, sb = 1;
  if (batch == 1) {
    const int64_t cus = ctx->num_cus > 0 ? ctx->num_cus : 256;
    sa = tiny_split(cus, ta + tb, a.R);
    if (b != nullptr) sb = tiny_split(cus, ta + tb, b->R);
  }
  // Split products reduce inside this launch (tiny_tile's FUSE) unless the
  // context asks for the separate launch; offsets of the partials at device
  // scope are 32-bit.
  bool fuse = false;
  if (sa > 1 || sb > 1) {
    const size_t na = sa > 1 ? (size_t)sa * a.P * a.Q : 0;
    const size_t nb = sb > 1 ? (size_t)sb * bb.P * bb.Q : 0;
    void *ws = nullptr;
    if (int rc = numrs_hip::workspace(ctx, (na + nb) * sizeof(float), &ws)) return rc;
    float *base = static_cast<float *>(ws);
    if (sa > 1) apply_splits(a, sa, base);
    if (sb > 1) apply_splits(bb, sb, base + na);
    fuse = ctx->split_reduce_mode == NUMRS_HIP_SPLIT_REDUCE_FUSED && 4 * (na + nb) < (size_t{1} << 31);
    if (fuse) {
      unsigned *cnt = nullptr;
      if (int rc = numrs_hip::arrival_counters(ctx, (size_t)(ta + tb), &cnt)) return rc;
      if (sa > 1) a.arrive = cnt;
      if (sb > 1) bb.arrive = cnt + ta;
    }
    ta *= sa;
    tb *= sb;
  }
  const dim3 grid((unsigned)(ta + tb + tc), (unsigned)batch);
  const ColSum c = cs != nullptr ? *cs : ColSum{};
  const int most_r = std::max(a.R, b != nullptr ? b->R : 0);
  auto go = [&](auto U, auto fuse_t) {
    constexpr int kU = decltype(U)::value;
    constexpr bool kF = decltype(fuse_t)::value;
    if (xa && ya)
      tiny_gemm_kernel<true, true, kU, kF><<<grid, kTinyThreads, 0, ctx->stream>>>(a, bb, (int)ta,
                                                                                    (int)tb, c);
    else if (xa)
      tiny_gemm_kernel<true, false, kU, kF><<<grid, kTinyThreads, 0, ctx->stream>>>(a, bb, (int)ta,
                                                                                     (int)tb, c);
    else if (ya)
      tiny_gemm_kernel<false, true, kU, kF><<<grid, kTinyThreads, 0, ctx->stream>>>(a, bb, (int)ta,
                                                                                     (int)tb, c);
    else
      tiny_gemm_kernel<false, false, kU, kF><<<grid, kTinyThreads, 0, ctx->stream>>>(a, bb, (int)ta,
                                                                                      (int)tb, c);
  };
  if (fuse)
    go(std::integral_constant<int, kTinyUSmall>{}, std::true_type{});
  else if (most_r > 16 * kTinyWaves * kTinyUSmall && sa == 1 && sb == 1)
    go(std::integral_constant<int, kTinyUBig>{}, std::false_type{});
  else
    go(std::integral_constant<int, kTinyUSmall>{}, std::false_type{});
  if (int rc = numrs_hip::check_launch(ctx, "tiny_gemm_kernel")) return rc;
  if (fuse) return NUMRS_HIP_OK;
  return reduce_splits(ctx, sa > 1 ? &a : nullptr, sb > 1 ? &bb : nullptr);
}

// ---------------------------------------------------------------------------
// Tile and split-K plan.  Model, from MI355X timings of grids of exactly 1..4
// tiles per CU at R = 256 and 1024 (NT, N(0, 1) data): `k` tiles of a shape
// resident on a CU take T steps (of 32) at step[k] us plus fixed[k] us
// (launch, pipeline fill, epilogue); a grid of W tiles puts ceil(W / CUs) on
// the busiest CU, in rounds of `most`.  A split product also writes and
// re-reads its fp32 partials (8 bytes per element per split) and launches
// splitk_reduce.
//   us at R = 256 | 1024: L, one: 33.1 | 98.5; M, one: 20.4 | 53.9; N, one:
//   15.5 | 41.6, two: 24.4 | 66.5; S, one: 10.6 | 27.3, two: 15.6 | 41.7,
//   three: 20.3 | 53.8.
struct ShapeInfo {
  int tp, tq, most;
  bool wide;
  double step[4], fixed[4];
};
enum { kL = 0, kM = 1, kN = 2, kS = 3, kShapeCount = 4 };
constexpr ShapeInfo kShapes[kShapeCount] = {
    {ShapeL::TP, ShapeL::TQ, 1, false, {0, 2.73}, {0, 11.3}},
    {ShapeM::TP, ShapeM::TQ, 1, false, {0, 1.45}, {0, 8.0}},
    {ShapeN::TP, ShapeN::TQ, 2, false, {0, 1.09, 1.75}, {0, 6.8, 10.4}},
    {ShapeS::TP, ShapeS::TQ, 3, true, {0, 0.70, 1.09, 1.40}, {0, 5.0, 6.9, 9.1}},
};
constexpr double kPartialBytesPerUs = 6.0e6, kReduceUs = 4.0;
constexpr int kMaxSplits = 32;

// Calls f with the shape's type.
template <typename F>
void with_shape(int shape, F &&f) {
  switch (shape) {
    case kL: return f(ShapeL{});
    case kM: return f(ShapeM{});
    case kN: return f(ShapeN{});
    default: return f(ShapeS{});
  }
}

// Whether the shape's loaders take both operands of g.
bool shape_fits(const Gemm &g, bool xrc, bool yrc, int shape) {
  constexpr int64_t kNarrow = int64_t{1} << 24;  // 32-bit offsets of up to 256 rows
  if (!kShapes[shape].wide && (g.ldx >= kNarrow || g.ldy >= kNarrow)) return false;
  bool ok = false;
  with_shape(shape, [&](auto s) {
    using S = decltype(s);
    ok = S::pairs_fit(xrc, g.P, S::TP) && S::pairs_fit(yrc, g.Q, S::TQ);
  });
  return ok;
}

double shape_us(const ShapeInfo &s, int64_t n, int T) {
  // most is 1, 2 or 3: no division by a variable
  const int64_t full = s.most == 1 ? n : s.most == 2 ? n / 2 : n / 3, left = n - full * s.most;
  double t = (double)full * ((double)T * s.step[s.most] + s.fixed[s.most]);
  if (left) t += (double)T * s.step[left] + s.fixed[left];
  return t;
}

struct Plan {
  int shape, sa, sb;
  double t;
};

template <typename T>
T ceil_div(T a, T b) {
  return (a + b - 1) / b;
}

// k tiles cut into ranges of at most T, of at most kMaxSplits: their number and length.
struct Cut {
  int n, len;
};
Cut cut(int k, int T) {
  const int len = ceil_div(k, std::min(ceil_div(k, T), kMaxSplits));
  return {ceil_div(k, len), len};
}

// Plan for a product a, or a pair with the TN product b in the same grid,
// over `batch` batch entries, all cut alike.  Candidate tile lengths T are
// ceil(k / s) for s = 1..kMaxSplits of either product; each product is cut
// into ceil(k / T) ranges (none empty) and the smallest estimate wins, ties
// going to the larger tile.  This is host time of every call, so lengths that
// repeat are passed over, and shapes whose steps alone, evenly over the CUs,
// take longer than the best plan so far (a pair 10.2 -> 0.9-2.0 us, a product
// 3.3 -> 0.5; the same plans).
Plan plan_product(numrs_hip_ctx *ctx, const Gemm &a, bool xa, bool ya, const Gemm *b,
                  int64_t batch) {
  const int64_t cus = std::max(ctx->num_cus, 1);
  Plan best{-1, 1, 1, 0.0};
  const int ka = ceil_div(a.R, kBR), kb = b ? ceil_div(b->R, kBR) : 0;
  const double pa = 8.0 * batch * a.P * a.Q / kPartialBytesPerUs;  // a split's partials
  const double pb = b ? 8.0 * batch * b->P * b->Q / kPartialBytesPerUs : 0.0;
  for (int shape = 0; shape < kShapeCount; ++shape) {
    if (!shape_fits(a, xa, ya, shape) || (b && !shape_fits(*b, false, false, shape))) continue;
    const ShapeInfo &s = kShapes[shape];
    const int64_t ta = (int64_t)ceil_div(a.P, s.tp) * ceil_div(a.Q, s.tq) * batch;
    const int64_t tb = b ? (int64_t)ceil_div(b->P, s.tp) * ceil_div(b->Q, s.tq) * batch : 0;
    double rate = s.step[1];  // of a tile and step, at best
    for (int n = 2; n <= s.most; ++n) rate = std::min(rate, s.step[n] / n);
    const double least = ((double)ta * ka + (double)tb * kb) / cus * rate;
    if (best.shape >= 0 && least * 0.999 > best.t) continue;
    for (int k : {ka, kb}) {
      for (int c = 1, last = 0; c <= kMaxSplits && k > 0; ++c) {
        const int T = ceil_div(k, c);
        if (T == last) continue;
        last = T;
        const Cut ca = cut(ka, T), cb = b ? cut(kb, T) : Cut{1, 0};
        const int64_t w = ta * ca.n + tb * cb.n;
        const int64_t n = w <= 0x7fffffff ? (int64_t)ceil_div((uint32_t)w, (uint32_t)cus) : ceil_div(w, cus);
        double t = shape_us(s, n, std::max(ca.len, cb.len));
        if (ca.n > 1) t += ca.n * pa;
        if (cb.n > 1) t += cb.n * pb;
        if (ca.n > 1 || cb.n > 1) t += kReduceUs;
        if (best.shape < 0 || t < best.t) best = {shape, ca.n, cb.n, t};
      }
    }
  }
  return best;  // S fits every product
}

// g as the plan's shape runs it.
Gemm as_shape(Gemm g, int shape) {
  g.tiles_p = ceil_div(g.P, kShapes[shape].tp);
  g.tiles_q = ceil_div(g.Q, kShapes[shape].tq);
  g.splits = 1;
  g.ktiles_per_split = ceil_div(g.R, kBR);
  g.partial = nullptr;
  return g;
}

// Descriptors for a plan, with split products pointed at the context's workspace.
// `sums`: room for the partial row sums of a split gb too (gb->sums).  A batch whose workspace is
// refused (no memory, or a recording that must not grow it) runs unsplit.
int prepare_plan(numrs_hip_ctx *ctx, const Plan &pl, int64_t batch, Gemm &ga, Gemm *gb, bool sums = false) {
  ga = as_shape(ga, pl.shape);
  if (gb != nullptr) *gb = as_shape(*gb, pl.shape);
  const size_t na = pl.sa > 1 ? (size_t)batch * pl.sa * ga.P * ga.Q : 0;
  const size_t nb = gb != nullptr && pl.sb > 1 ? (size_t)batch * pl.sb * gb->P * gb->Q : 0;
  if (na + nb == 0) return NUMRS_HIP_OK;
  void *ws = nullptr;
  const size_t at = (na + nb + 3) & ~size_t{3}, ns = sums && nb ? (size_t)pl.sb * gb->P : 0;
  if (int rc = numrs_hip::workspace(ctx, (at + ns) * sizeof(float), &ws)) {
    if (batch == 1) return rc;
    (void)hipGetLastError();
    return NUMRS_HIP_OK;
  }
  float *base = static_cast<float *>(ws);
  if (ns) gb->sums = base + at;
  if (na) apply_splits(ga, pl.sa, base);
  if (nb) apply_splits(*gb, pl.sb, base + na);
  return NUMRS_HIP_OK;
}

int64_t grid_tiles(const Gemm &g) { return (int64_t)g.tiles_p * g.tiles_q * g.splits; }

int check_dims(numrs_hip_ctx *ctx, const char *who, int64_t batch, int64_t M, int64_t K,
               int64_t N) {
  if (batch < 0 || M < 0 || K < 0 || N < 0)
    return numrs_hip::fail(ctx, NUMRS_HIP_E_INVALID, "%s: negative dimension", who);
  const int64_t lim = (int64_t)1 << 30;
  if (M >= lim || K >= lim || N >= lim || batch >= 65536)
    return numrs_hip::fail(ctx, NUMRS_HIP_E_INVALID, "%s: dimension too large", who);
  return NUMRS_HIP_OK;
}

Gemm make(const float *X, const float *Y, float *C, int64_t ldx, int64_t ldy, int64_t ldc,
          int64_t bsx, int64_t bsy, int64_t bsc, int64_t P, int64_t Q, int64_t R, int acc) {
  Gemm g;
  g.X = X;
  g.Y = Y;
  g.C = C;
  g.ldx = ldx;
  g.ldy = ldy;
  g.ldc = ldc;
  g.bsx = bsx;
  g.bsy = bsy;
  g.bsc = bsc;
  g.bsx2 = g.bsy2 = g.bsc2 = 0;
  g.binner = 1;
  g.alpha = 1.0f;
  g.splits = 1;
  g.ktiles_per_split = (int)((R + kBR - 1) / kBR);
  g.partial = nullptr;
  g.bias = nullptr;
  g.xmask = nullptr;
  g.act = 0;
  g.pre = nullptr;
  g.res = nullptr;
  g.ldr = 0;
  g.arrive = nullptr;
  g.sums = nullptr;
  g.sums_acc = 0;
  g.P = (int)P;
  g.Q = (int)Q;
  g.R = (int)R;
  g.tiles_p = g.tiles_q = 0;  // as_shape
  g.accumulate = acc;
  return g;
}

// Zero-length reduction: C = 0 (or unchanged when accumulating).
int zero_output(numrs_hip_ctx *ctx, float *C, int64_t count, int acc) {
  if (acc || count == 0) return NUMRS_HIP_OK;
  return numrs_hip_fill(ctx, C, count, 0.0f);
}

template <bool XRC, bool YRC>
int launch_one(numrs_hip_ctx *ctx, Gemm g, int64_t batch) {
  if (g.P == 0 || g.Q == 0 || batch == 0) return NUMRS_HIP_OK;
  if (tiny_fits(g, batch)) return launch_tiny(ctx, g, XRC, YRC, nullptr, batch, nullptr);
  const Plan pl = plan_product(ctx, g, XRC, YRC, nullptr, batch);
  if (int rc = prepare_plan(ctx, pl, batch, g, nullptr)) return rc;
  if (grid_tiles(g) * batch > 0x7fffffff)
    return numrs_hip::fail(ctx, NUMRS_HIP_E_INVALID, "gemm: too many tiles");
  const dim3 grid((unsigned)grid_tiles(g), (unsigned)batch);
  if (g.act && g.splits == 1) {  // activation in the tile epilogue (the Linear forward)
    if constexpr (XRC && YRC) {
      with_shape(pl.shape, [&](auto s) {
        using S = decltype(s);
        gemm_kernel<true, true, S, true><<<grid, S::NT, 0, ctx->stream>>>(g);
      });
    } else {
      return numrs_hip::fail(ctx, NUMRS_HIP_E_INVALID, "gemm: activation on a non-NT product");
    }
  } else {
    with_shape(pl.shape, [&](auto s) {
      using S = decltype(s);
      gemm_kernel<XRC, YRC, S><<<grid, S::NT, 0, ctx->stream>>>(g);
    });
  }
  if (int rc = numrs_hip::check_launch(ctx, "gemm_kernel")) return rc;
  return reduce_splits(ctx, &g, nullptr, nullptr, nullptr, batch);
}

// One launch of the products ga (layout xa, ya: NT, NN or TN) and gb (TN),
// then the reduction of their splits with the column sums cs and the set
// extra (reduce_splits).  `sums` (NN + TN, batch 1): column sums of gb's X,
// formed by its tiles; split, their partials are added in order by the same
// reduction (plainly: a compensated sum makes NaN of an infinity).
int launch_two(numrs_hip_ctx *ctx, Gemm ga, bool xa, bool ya, Gemm gb, int64_t batch,
               const ColSum *cs, const SplitSet *extra, const char *who,
               const ColSum *sums = nullptr) {
  const Plan pl = plan_product(ctx, ga, xa, ya, &gb, batch);
  if (sums != nullptr) gb.sums = sums->out, gb.sums_acc = sums->acc;
  if (int rc = prepare_plan(ctx, pl, batch, ga, &gb, sums != nullptr)) return rc;
  SplitSet part;
  if (sums != nullptr && gb.splits > 1) {
    part = SplitSet{gb.sums, sums->out, nullptr, gb.P, gb.P, gb.P, gb.splits, sums->acc, 1.0f, 0,
                    nullptr, nullptr, 0, 0, 0, 0, 1};
    gb.sums_acc = 0;
    extra = &part;
  }
  const int64_t na = grid_tiles(ga), total = na + grid_tiles(gb);
  if (total * batch > 0x7fffffff)
    return numrs_hip::fail(ctx, NUMRS_HIP_E_INVALID, "%s: too large", who);
  const dim3 grid((unsigned)total, (unsigned)batch);
  with_shape(pl.shape, [&](auto s) {
    using S = decltype(s);
    if (sums != nullptr)
      gemm_pair_kernel<true, false, S, true><<<grid, S::NT, 0, ctx->stream>>>(ga, gb, (int)na);
    else if (xa && ya)
      gemm_pair_kernel<true, true, S><<<grid, S::NT, 0, ctx->stream>>>(ga, gb, (int)na);
    else if (xa)
      gemm_pair_kernel<true, false, S><<<grid, S::NT, 0, ctx->stream>>>(ga, gb, (int)na);
    else
      gemm_pair_kernel<false, false, S><<<grid, S::NT, 0, ctx->stream>>>(ga, gb, (int)na);
  });
  if (int rc = numrs_hip::check_launch(ctx, who)) return rc;
  return reduce_splits(ctx, &ga, &gb, cs, extra, batch);
}

int gemm_dispatch(numrs_hip_ctx *ctx, const Gemm &g, int64_t batch, bool xrc, bool yrc) {
  if (xrc && yrc) return launch_one<true, true>(ctx, g, batch);
  if (xrc && !yrc) return launch_one<true, false>(ctx, g, batch);
  if (!xrc && yrc) return launch_one<false, true>(ctx, g, batch);
  return launch_one<false, false>(ctx, g, batch);
}

int matmul_backward_impl(numrs_hip_ctx *ctx, const float *dC, const float *A, const float *B,
                         float *dA, float *dB, int64_t batch, int64_t M, int64_t K, int64_t N,
                         int64_t sa, int64_t sb, int64_t sc, int acc) {
  const char *who = "numrs_hip_matmul_backward";
  int rc = check_dims(ctx, who, batch, M, K, N);
  if (rc) return rc;
  if (dA == nullptr && dB == nullptr) return NUMRS_HIP_OK;
  if (batch == 0 || M == 0 || K == 0 || N == 0) {
    // Empty operands (0-byte buffers may be NULL): dA is reduced over N and dB
    // over M, so an empty reduction dimension gives zero gradients.
    for (int64_t b = 0; b < batch; ++b) {
      if (dA && M * K > 0) rc = zero_output(ctx, dA + b * sa, M * K, acc);
      if (!rc && dB && K * N > 0) rc = zero_output(ctx, dB + b * sb, K * N, acc);
      if (rc) return rc;
    }
    return NUMRS_HIP_OK;
  }
  if (dC == nullptr || (dA != nullptr && B == nullptr) || (dB != nullptr && A == nullptr))
    return numrs_hip::fail(ctx, NUMRS_HIP_E_INVALID, "%s: null input pointer", who);
  // dA[M,K] = dC[M,N] @ B[K,N]^T : P=M, Q=K, R=N, X=dC (ld N), Y=B (ld N)
  Gemm ga = make(dC, B, dA, N, N, K, sc, sb, sa, M, K, N, acc);
  // dB[K,N] = A[M,K]^T @ dC[M,N] : P=K, Q=N, R=M, X=A (ld K), Y=dC (ld N)
  Gemm gb = make(A, dC, dB, K, N, N, sa, sc, sb, K, N, M, acc);
  if (dA == nullptr) return gemm_dispatch(ctx, gb, batch, false, false);
  if (dB == nullptr) return gemm_dispatch(ctx, ga, batch, true, true);
  if (tiny_fits(ga, batch) && tiny_fits(gb, batch))
    return launch_tiny(ctx, ga, true, true, &gb, batch, nullptr);
  return launch_two(ctx, ga, true, true, gb, batch, nullptr, nullptr, who);
}

int matmul_impl(numrs_hip_ctx *ctx, const float *A, const float *B, float *C, int64_t batch,
                int64_t M, int64_t K, int64_t N, int64_t sa, int64_t sb, int64_t sc, int ta,
                int tb, int acc) {
  const char *who = "numrs_hip_matmul";
  int rc = check_dims(ctx, who, batch, M, K, N);
  if (rc) return rc;
  if (batch == 0 || M == 0 || N == 0) return NUMRS_HIP_OK;
  if (C == nullptr || ((A == nullptr || B == nullptr) && K > 0))
    return numrs_hip::fail(ctx, NUMRS_HIP_E_INVALID, "%s: null pointer", who);
  if (K == 0) {
    for (int64_t b = 0; b < batch; ++b)
      if ((rc = zero_output(ctx, C + b * sc, M * N, acc))) return rc;
    return NUMRS_HIP_OK;
  }
  // op(A)[M,K]: R-contiguous unless transposed (stored [K,M]).
  const bool xrc = !ta;
  const int64_t ldx = ta ? M : K;
  // op(B)[K,N]: Q-contiguous unless transposed (stored [N,K], R-contiguous).
  const bool yrc = tb != 0;
  const int64_t ldy = tb ? K : N;
  Gemm g = make(A, B, C, ldx, ldy, N, sa, sb, sc, M, N, K, acc);
  return gemm_dispatch(ctx, g, batch, xrc, yrc);
}

int gemm_general(numrs_hip_ctx *ctx, const float *A, int64_t lda, const float *B, int64_t ldb,
                 float *C, int64_t ldc, int64_t M, int64_t K, int64_t N, int ta, int tb,
                 float alpha, int acc, int64_t batch, int64_t binner, int64_t sao, int64_t sai,
                 int64_t sbo, int64_t sbi, int64_t sco, int64_t sci) {
  const char *who = "numrs_hip_gemm";
  int rc = check_dims(ctx, who, batch, M, K, N);
  if (rc) return rc;
  if (binner < 1 || binner > batch + (batch == 0))
    return numrs_hip::fail(ctx, NUMRS_HIP_E_INVALID, "%s: batch_inner %lld", who, (long long)binner);
  if (lda < 0 || ldb < 0 || ldc < N || sao < 0 || sai < 0 || sbo < 0 || sbi < 0 || sco < 0 ||
      sci < 0)
    return numrs_hip::fail(ctx, NUMRS_HIP_E_INVALID, "%s: bad leading dimension or stride", who);
  if (lda < (ta ? M : K) || ldb < (tb ? K : N))
    return numrs_hip::fail(ctx, NUMRS_HIP_E_INVALID, "%s: leading dimension too small", who);
  if (batch == 0 || M == 0 || N == 0) return NUMRS_HIP_OK;
  if (C == nullptr || ((A == nullptr || B == nullptr) && K > 0))
    return numrs_hip::fail(ctx, NUMRS_HIP_E_INVALID, "%s: null pointer", who);
  Gemm g = make(A, B, C, lda, ldb, ldc, sao, sbo, sco, M, N, K, acc);
  g.bsx2 = sai;
  g.bsy2 = sbi;
  g.bsc2 = sci;
  g.binner = (int)binner;
  g.alpha = alpha;
  if (K == 0) {
    if (acc) return NUMRS_HIP_OK;
    if (ldc != N || binner != 1 || sco != M * N)
      return numrs_hip::fail(ctx, NUMRS_HIP_E_INVALID, "%s: empty reduction into a strided C", who);
    return numrs_hip_fill(ctx, C, batch * M * N, 0.0f);
  }
  return gemm_dispatch(ctx, g, batch, !ta, tb != 0);
}

// Launches a (first, TN-second) product pair in one grid with per-product
// split-K; `first_nt` selects the NT (matmul_backward dA) or NN (Linear dx)
// layout of the first product.  Either product may be absent (C == null).
// `cs` (optional): column sums that the pair's launch forms too -- the tiny
// kernel's own workgroups; of the second product's own X (a Linear's bias
// gradient), its tiles; else the split-reduce launch (a launch of its own
// when neither product is split) where colsum_fits.  *cs_done says whether
// they were formed.
int launch_pair(numrs_hip_ctx *ctx, Gemm ga, Gemm gb, bool first_nt, const char *who,
                const ColSum *cs_in = nullptr, bool *cs_done = nullptr) {
  const bool has_a = ga.C != nullptr, has_b = gb.C != nullptr;
  if (cs_done != nullptr) *cs_done = false;
  if ((has_a || has_b) && (!has_a || tiny_fits(ga, 1)) && (!has_b || tiny_fits(gb, 1)) &&
      (cs_in == nullptr || cs_in->rows <= kTinyColsumRows)) {
    if (cs_done != nullptr) *cs_done = cs_in != nullptr;
    if (has_a) return launch_tiny(ctx, ga, true, first_nt, has_b ? &gb : nullptr, 1, cs_in);
    return launch_tiny(ctx, gb, false, false, nullptr, 1, cs_in);
  }
  if (has_a && has_b && !first_nt && cs_in != nullptr && cs_in->mask == nullptr && cs_in->g == gb.X &&
      cs_in->ldg == gb.ldx && cs_in->rows == gb.R && cs_in->cols == gb.P) {
    if (cs_done != nullptr) *cs_done = true;
    return launch_two(ctx, ga, true, false, gb, 1, nullptr, nullptr, who, cs_in);
  }
  const ColSum *cs = cs_in != nullptr && cs_in->mask == nullptr &&
                             colsum_fits(cs_in->g, cs_in->rows, cs_in->cols, cs_in->ldg)
                         ? cs_in
                         : nullptr;
  if (cs_done != nullptr) *cs_done = cs != nullptr;
  if (!has_a && !has_b) return cs ? reduce_splits(ctx, nullptr, nullptr, cs) : NUMRS_HIP_OK;
  if (!has_a || !has_b) {
    if (int rc = has_a ? gemm_dispatch(ctx, ga, 1, true, first_nt)
                       : gemm_dispatch(ctx, gb, 1, false, false))
      return rc;
    return cs ? reduce_splits(ctx, nullptr, nullptr, cs) : NUMRS_HIP_OK;
  }
  return launch_two(ctx, ga, true, first_nt, gb, 1, cs, nullptr, who);
}

}  // namespace

int numrs_hip::gemm_nn_tn_pair(numrs_hip_ctx *ctx, BatchedMat X, BatchedMat Y1, BatchedOut C1,
                               BatchedMat Y2, BatchedOut C2, int64_t M, int64_t K, int64_t N,
                               float alpha, int accumulate, int64_t batch, int64_t binner) {
  const char *who = "gemm_nn_tn_pair";
  if (int rc = check_dims(ctx, who, batch, M, K, N)) return rc;
  if (binner < 1 || binner > std::max<int64_t>(batch, 1))
    return numrs_hip::fail(ctx, NUMRS_HIP_E_INVALID, "%s: batch_inner %lld", who, (long long)binner);
  if (batch == 0 || N == 0 || (C1.p == nullptr && C2.p == nullptr)) return NUMRS_HIP_OK;
  // C1[M,N] = X[M,K] Y1[K,N]: P=M, Q=N, R=K, X reduction-contiguous.
  Gemm ga = make(X.p, Y1.p, C1.p, X.ld, Y1.ld, C1.ld, X.so, Y1.so, C1.so, M, N, K, accumulate);
  // C2[K,N] = X^T Y2[M,N]: P=K, Q=N, R=M, X output-contiguous.
  Gemm gb = make(X.p, Y2.p, C2.p, X.ld, Y2.ld, C2.ld, X.so, Y2.so, C2.so, K, N, M, accumulate);
  ga.bsx2 = X.si, ga.bsy2 = Y1.si, ga.bsc2 = C1.si;
  gb.bsx2 = X.si, gb.bsy2 = Y2.si, gb.bsc2 = C2.si;
  ga.binner = gb.binner = (int)binner;
  ga.alpha = gb.alpha = alpha;
  if (M == 0 || K == 0) {
    // an empty reduction leaves zeros (or the accumulated values)
    for (int64_t z = 0; z < batch && !accumulate; ++z) {
      const int64_t zo = z / binner, zi = z - zo * binner;
      if (C1.p && M > 0)
        for (int64_t r = 0; r < M; ++r)
          if (int rc = numrs_hip_fill(ctx, C1.p + zo * C1.so + zi * C1.si + r * C1.ld, N, 0.0f))
            return rc;
      if (C2.p && K > 0)
        for (int64_t r = 0; r < K; ++r)
          if (int rc = numrs_hip_fill(ctx, C2.p + zo * C2.so + zi * C2.si + r * C2.ld, N, 0.0f))
            return rc;
    }
    return NUMRS_HIP_OK;
  }
  if (X.p == nullptr || (C1.p && Y1.p == nullptr) || (C2.p && Y2.p == nullptr))
    return numrs_hip::fail(ctx, NUMRS_HIP_E_INVALID, "%s: null input", who);
  if (C1.p == nullptr) return gemm_dispatch(ctx, gb, batch, false, false);
  if (C2.p == nullptr) return gemm_dispatch(ctx, ga, batch, true, false);
  if (batch == 1) return launch_pair(ctx, ga, gb, false, who);
  if (tiny_fits(ga, batch) && tiny_fits(gb, batch))
    return launch_tiny(ctx, ga, true, false, &gb, batch, nullptr);
  return launch_two(ctx, ga, true, false, gb, batch, nullptr, nullptr, who);
}

int numrs_hip::gemm_tn2_colsum(numrs_hip_ctx *ctx, const float *X, int64_t ldx, int64_t M,
                               int64_t K, const float *Y1, int64_t ldy1, int64_t N1, float *C1,
                               int acc1, const float *Y2, int64_t ldy2, int64_t N2, float *C2,
                               int acc2, float *db, int acc_db, const float *db_part,
                               int64_t db_rows) {
  const char *who = "gemm_tn2_colsum";
  if (int rc = check_dims(ctx, who, 1, M, K, std::max(N1, N2))) return rc;
  if (X == nullptr || C1 == nullptr || C2 == nullptr || Y1 == nullptr || Y2 == nullptr ||
      M <= 0 || K <= 0 || N1 <= 0 || N2 <= 0)
    return numrs_hip::fail(ctx, NUMRS_HIP_E_INVALID, "%s: null or empty operand", who);
  // C[K,N] = X^T Y with X [M,K], Y [M,N]: P=K, Q=N, R=M (both operands
  // output-contiguous).
  Gemm ga = make(X, Y1, C1, ldx, ldy1, N1, 0, 0, 0, K, N1, M, acc1);
  Gemm gb = make(X, Y2, C2, ldx, ldy2, N2, 0, 0, 0, K, N2, M, acc2);
  ColSum cs{X, db, M, K, ldx, acc_db, nullptr};
  // db from row partials: the compensated sum over db_rows rows of db_part
  // [db_rows, K] in row order, as one more set of the split reduce
  const bool by_part = db != nullptr && db_part != nullptr && db_rows >= 1 && db_rows <= (1 << 20);
  SplitSet part{db_part, db, nullptr, K, K, (int)K, (int)db_rows, acc_db, 1.0f, 0, nullptr,
                nullptr, 0, 1, 0, 0, 1};
  const SplitSet *extra = by_part ? &part : nullptr;
  const bool cs_ok = db != nullptr && !by_part && colsum_fits(X, M, K, ldx);
  if (tiny_fits(ga, 1) && tiny_fits(gb, 1)) {
    if (int rc = launch_tiny(ctx, ga, false, false, &gb, 1, nullptr)) return rc;
    if (cs_ok || by_part)
      if (int rc = reduce_splits(ctx, nullptr, nullptr, cs_ok ? &cs : nullptr, extra)) return rc;
  } else if (int rc = launch_two(ctx, ga, false, false, gb, 1, cs_ok ? &cs : nullptr, extra, who)) {
    return rc;
  }
  if (db == nullptr || cs_ok || by_part) return NUMRS_HIP_OK;
  const int64_t gs[2] = {M, K};
  return numrs_hip_sum_to_shape(ctx, X, gs, 2, db, &K, 1, NUMRS_HIP_UNBROADCAST_CORRECT, acc_db);
}

extern "C" {

int numrs_hip_set_split_reduction(numrs_hip_ctx *ctx, int mode) {
  NRS_CHECK_CTX(ctx);
  if (mode != NUMRS_HIP_SPLIT_REDUCE_FUSED && mode != NUMRS_HIP_SPLIT_REDUCE_SEPARATE)
    return numrs_hip::fail(ctx, NUMRS_HIP_E_INVALID, "split reduction mode %d", mode);
  ctx->split_reduce_mode = mode;
  return NUMRS_HIP_OK;
}

int numrs_hip_linear_forward(numrs_hip_ctx *ctx, const float *x, const float *W, const float *b,
                             float *y, int64_t T, int64_t in, int64_t out) {
  NRS_CHECK_CTX(ctx);
  const char *who = "numrs_hip_linear_forward";
  if (int rc = check_dims(ctx, who, 1, T, in, out)) return rc;
  if (T == 0 || out == 0) return NUMRS_HIP_OK;
  if (y == nullptr || (in > 0 && (x == nullptr || W == nullptr)))
    return numrs_hip::fail(ctx, NUMRS_HIP_E_INVALID, "%s: null pointer", who);
  if (in == 0) {  // empty product: y = b broadcast over rows (or 0)
    if (int rc = numrs_hip_fill(ctx, y, T * out, 0.0f)) return rc;
    if (b == nullptr) return NUMRS_HIP_OK;
    const int64_t bs = out;
    const int64_t ys[2] = {T, out};
    return numrs_hip_binary_forward(ctx, NUMRS_HIP_ADD, y, ys, 2, b, &bs, 1, y);
  }
  // y[T,out] = x[T,in] @ W[out,in]^T + b : X = x (R-contig), Y = W^T (R-contig)
  Gemm g = make(x, W, y, in, in, out, 0, 0, 0, T, out, in, 0);
  g.bias = b;
  return gemm_dispatch(ctx, g, 1, true, true);
}

int numrs_hip_linear_backward(numrs_hip_ctx *ctx, const float *g, const float *x, const float *W,
                              float *dx, float *dW, float *db, int64_t T, int64_t in, int64_t out,
                              int acc_dx, int acc_dw, int acc_db, int mode) {
  NRS_CHECK_CTX(ctx);
  const char *who = "numrs_hip_linear_backward";
  if (int rc = check_dims(ctx, who, 1, T, in, out)) return rc;
  if (g == nullptr || (dx && W == nullptr) || (dW && x == nullptr))
    return numrs_hip::fail(ctx, NUMRS_HIP_E_INVALID, "%s: null input", who);
  if (T == 0 || out == 0) {  // empty reductions: zero gradients
    if (dx && !acc_dx && T * in > 0)
      if (int rc = numrs_hip_fill(ctx, dx, T * in, 0.0f)) return rc;
    if (dW && !acc_dw && out * in > 0)
      if (int rc = numrs_hip_fill(ctx, dW, out * in, 0.0f)) return rc;
  } else {
    // db = column sums of g (CORRECT mode), formed by the pair's own launch
    // (launch_pair: tiny products' own workgroups, or the dW product's tiles)
    // or, without dx or dW, by a launch of their own
    ColSum cs{g, db, T, out, out, acc_db};
    const bool want_db = db != nullptr && mode == NUMRS_HIP_UNBROADCAST_CORRECT;
    bool db_done = false;
    if (in > 0) {
      // dx[T,in] = g[T,out] @ W[out,in] : X = g (R-contig), Y = W (Q-contig)  [NN]
      Gemm gx = make(g, W, dx, out, in, in, 0, 0, 0, T, in, out, acc_dx);
      // dW[out,in] = g^T @ x : X = g^T (P-contig), Y = x (Q-contig)          [TN]
      Gemm gw = make(g, x, dW, out, in, in, 0, 0, 0, out, in, T, acc_dw);
      if (int rc = launch_pair(ctx, gx, gw, false, who, want_db ? &cs : nullptr, &db_done))
        return rc;
    } else if (want_db && colsum_fits(g, T, out, out)) {
      if (int rc = reduce_splits(ctx, nullptr, nullptr, &cs)) return rc;
      db_done = true;
    }
    if (db_done) return NUMRS_HIP_OK;
  }
  if (db == nullptr || out == 0) return NUMRS_HIP_OK;
  const int64_t gs[2] = {T, out};
  const int64_t bs = out;
  return numrs_hip_sum_to_shape(ctx, g, gs, 2, db, &bs, 1, mode, acc_db);
}

int numrs_hip_linear_relu_forward(numrs_hip_ctx *ctx, const float *x, const float *W,
                                  const float *b, float *y, int64_t T, int64_t in, int64_t out) {
  NRS_CHECK_CTX(ctx);
  const char *who = "numrs_hip_linear_relu_forward";
  if (int rc = check_dims(ctx, who, 1, T, in, out)) return rc;
  if (T == 0 || out == 0) return NUMRS_HIP_OK;
  if (y == nullptr || (in > 0 && (x == nullptr || W == nullptr)))
    return numrs_hip::fail(ctx, NUMRS_HIP_E_INVALID, "%s: null pointer", who);
  if (in == 0) {  // empty product: ReLU of the broadcast bias
    if (int rc = numrs_hip_linear_forward(ctx, x, W, b, y, T, in, out)) return rc;
    return numrs_hip_unary_forward(ctx, NUMRS_HIP_RELU, y, y, T * out, 0.0f);
  }
  Gemm g = make(x, W, y, in, in, out, 0, 0, 0, T, out, in, 0);
  g.bias = b;
  g.act = kActRelu;
  return gemm_dispatch(ctx, g, 1, true, true);
}

int numrs_hip_linear_gelu_forward(numrs_hip_ctx *ctx, const float *x, const float *W,
                                  const float *b, float *y, float *pre, int64_t T, int64_t in,
                                  int64_t out) {
  NRS_CHECK_CTX(ctx);
  const char *who = "numrs_hip_linear_gelu_forward";
  if (int rc = check_dims(ctx, who, 1, T, in, out)) return rc;
  if (T == 0 || out == 0) return NUMRS_HIP_OK;
  if (y == nullptr || pre == nullptr || pre == y || (in > 0 && (x == nullptr || W == nullptr)))
    return numrs_hip::fail(ctx, NUMRS_HIP_E_INVALID, "%s: null or aliased pointer", who);
  if (in == 0) {  // empty product: GELU of the broadcast bias
    if (int rc = numrs_hip_linear_forward(ctx, x, W, b, pre, T, in, out)) return rc;
    return numrs_hip_unary_forward(ctx, NUMRS_HIP_GELU, pre, y, T * out, 0.0f);
  }
  Gemm g = make(x, W, y, in, in, out, 0, 0, 0, T, out, in, 0);
  g.bias = b;
  g.act = kActGelu;
  g.pre = pre;
  return gemm_dispatch(ctx, g, 1, true, true);
}

int numrs_hip_linear_gelu_backward(numrs_hip_ctx *ctx, const float *g, const float *pre,
                                   const float *x, const float *W, float *dx, float *dW,
                                   float *db, int64_t T, int64_t in, int64_t out, int acc_dx,
                                   int acc_dw, int acc_db, int mode) {
  NRS_CHECK_CTX(ctx);
  const char *who = "numrs_hip_linear_gelu_backward";
  if (int rc = check_dims(ctx, who, 1, T, in, out)) return rc;
  if (T == 0 || out == 0)
    return numrs_hip_linear_backward(ctx, g, x, W, dx, dW, db, T, in, out, acc_dx, acc_dw, acc_db,
                                     mode);
  if (g == nullptr || pre == nullptr)
    return numrs_hip::fail(ctx, NUMRS_HIP_E_INVALID, "%s: null input", who);
  // The pre-activation gradient g * GELU'(pre), then the Linear backward.
  numrs_hip::TempBlock gp(ctx);
  if (int rc = gp.alloc((size_t)T * out * sizeof(float))) return rc;
  if (int rc = numrs_hip_unary_backward(ctx, NUMRS_HIP_GELU, g, pre, gp.f(), T * out, 0.0f, 0))
    return rc;
  return numrs_hip_linear_backward(ctx, gp.f(), x, W, dx, dW, db, T, in, out, acc_dx, acc_dw,
                                   acc_db, mode);
}

int numrs_hip_linear_relu_backward(numrs_hip_ctx *ctx, const float *g, const float *y,
                                   const float *x, const float *W, float *dx, float *dW,
                                   float *db, int64_t T, int64_t in, int64_t out, int acc_dx,
                                   int acc_dw, int acc_db, int mode) {
  NRS_CHECK_CTX(ctx);
  const char *who = "numrs_hip_linear_relu_backward";
  if (int rc = check_dims(ctx, who, 1, T, in, out)) return rc;
  if (T == 0 || out == 0)  // empty reductions: the Linear backward's zero gradients
    return numrs_hip_linear_backward(ctx, g, x, W, dx, dW, db, T, in, out, acc_dx, acc_dw, acc_db,
                                     mode);
  if (g == nullptr || y == nullptr || (dx && W == nullptr) || (dW && x == nullptr))
    return numrs_hip::fail(ctx, NUMRS_HIP_E_INVALID, "%s: null input", who);
  if ((dx != nullptr || dW != nullptr) && in > 0 &&
      (db == nullptr || (mode == NUMRS_HIP_UNBROADCAST_CORRECT && T <= kTinyColsumRows))) {
    // The pre-activation gradient (y > 0 ? g : 0) applied as the tiny
    // kernel loads g: one launch for dx, dW and db.
    Gemm gx = make(g, W, dx, out, in, in, 0, 0, 0, T, in, out, acc_dx);
    Gemm gw = make(g, x, dW, out, in, in, 0, 0, 0, out, in, T, acc_dw);
    gx.xmask = gw.xmask = y;
    if ((dx == nullptr || tiny_fits(gx, 1)) && (dW == nullptr || tiny_fits(gw, 1))) {
      const ColSum cs{g, db, T, out, out, acc_db, y};
      const ColSum *csp = db != nullptr ? &cs : nullptr;
      if (dx != nullptr) return launch_tiny(ctx, gx, true, false, dW ? &gw : nullptr, 1, csp);
      return launch_tiny(ctx, gw, false, false, nullptr, 1, csp);
    }
  }
  // Otherwise the masked gradient first, then the Linear backward on it.
  if ((dx == nullptr && dW == nullptr) || in == 0) {
    if (int rc = numrs_hip_linear_backward(ctx, g, x, W, dx, dW, nullptr, T, in, out, acc_dx,
                                           acc_dw, 0, mode))
      return rc;
    return db ? numrs_hip_relu_bias_backward(ctx, g, y, nullptr, db, T, out, mode, acc_db)
              : NUMRS_HIP_OK;
  }
  numrs_hip::TempBlock gm(ctx);
  if (int rc = gm.alloc((size_t)T * out * sizeof(float))) return rc;
  if (int rc = numrs_hip_relu_bias_backward(ctx, g, y, gm.f(), nullptr, T, out, mode, 0))
    return rc;
  return numrs_hip_linear_backward(ctx, gm.f(), x, W, dx, dW, db, T, in, out, acc_dx, acc_dw,
                                   acc_db, mode);
}

int numrs_hip_linear_residual_forward(numrs_hip_ctx *ctx, const float *x, const float *W,
                                      const float *b, const float *res, float *y, int64_t T,
                                      int64_t in, int64_t out) {
  NRS_CHECK_CTX(ctx);
  const char *who = "numrs_hip_linear_residual_forward";
  if (int rc = check_dims(ctx, who, 1, T, in, out)) return rc;
  if (T == 0 || out == 0) return NUMRS_HIP_OK;
  if (y == nullptr || res == nullptr || (in > 0 && (x == nullptr || W == nullptr)))
    return numrs_hip::fail(ctx, NUMRS_HIP_E_INVALID, "%s: null pointer", who);
  if (in == 0) {  // empty product: y = b broadcast over rows (or 0), then + res
    if (int rc = numrs_hip_linear_forward(ctx, x, W, b, y, T, in, out)) return rc;
    const int64_t ys[2] = {T, out};
    return numrs_hip_binary_forward(ctx, NUMRS_HIP_ADD, res, ys, 2, y, ys, 2, y);
  }
  Gemm g = make(x, W, y, in, in, out, 0, 0, 0, T, out, in, 0);
  g.bias = b;
  g.res = res;
  g.ldr = out;
  return gemm_dispatch(ctx, g, 1, true, true);
}

int numrs_hip_gemm(numrs_hip_ctx *ctx, const float *A, int64_t lda, const float *B, int64_t ldb,
                   float *C, int64_t ldc, int64_t M, int64_t K, int64_t N, int trans_a,
                   int trans_b, float alpha, int accumulate, int64_t batch, int64_t batch_inner,
                   int64_t sa_outer, int64_t sa_inner, int64_t sb_outer, int64_t sb_inner,
                   int64_t sc_outer, int64_t sc_inner) {
  NRS_CHECK_CTX(ctx);
  return gemm_general(ctx, A, lda, B, ldb, C, ldc, M, K, N, trans_a, trans_b, alpha, accumulate,
                      batch, batch_inner, sa_outer, sa_inner, sb_outer, sb_inner, sc_outer,
                      sc_inner);
}

int numrs_hip_matmul_backward(numrs_hip_ctx *ctx, const float *dC, const float *A,
                              const float *B, float *dA, float *dB, int64_t M, int64_t K,
                              int64_t N, int accumulate) {
  NRS_CHECK_CTX(ctx);
  return matmul_backward_impl(ctx, dC, A, B, dA, dB, 1, M, K, N, 0, 0, 0, accumulate);
}

int numrs_hip_matmul_backward_batched(numrs_hip_ctx *ctx, const float *dC, const float *A,
                                      const float *B, float *dA, float *dB, int64_t batch,
                                      int64_t M, int64_t K, int64_t N, int64_t stride_a,
                                      int64_t stride_b, int64_t stride_c, int accumulate) {
  NRS_CHECK_CTX(ctx);
  if (stride_a < 0 || stride_b < 0 || stride_c < 0)
    return numrs_hip::fail(ctx, NUMRS_HIP_E_INVALID, "negative batch stride");
  return matmul_backward_impl(ctx, dC, A, B, dA, dB, batch, M, K, N, stride_a, stride_b,
                              stride_c, accumulate);
}

int numrs_hip_matmul(numrs_hip_ctx *ctx, const float *A, const float *B, float *C, int64_t M,
                     int64_t K, int64_t N, int trans_a, int trans_b, int accumulate) {
  NRS_CHECK_CTX(ctx);
  return matmul_impl(ctx, A, B, C, 1, M, K, N, 0, 0, 0, trans_a, trans_b, accumulate);
}

int numrs_hip_matmul_batched(numrs_hip_ctx *ctx, const float *A, const float *B, float *C,
                             int64_t batch, int64_t M, int64_t K, int64_t N, int64_t stride_a,
                             int64_t stride_b, int64_t stride_c, int trans_a, int trans_b,
                             int accumulate) {
  NRS_CHECK_CTX(ctx);
  if (stride_a < 0 || stride_b < 0 || stride_c < 0)
    return numrs_hip::fail(ctx, NUMRS_HIP_E_INVALID, "negative batch stride");
  return matmul_impl(ctx, A, B, C, batch, M, K, N, stride_a, stride_b, stride_c, trans_a,
                     trans_b, accumulate);
}

}  // extern "C"
