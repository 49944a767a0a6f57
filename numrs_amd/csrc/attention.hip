// Multi-head attention forward / backward for the transformer configuration
// (no reference op: numrs has no attention and a 2-D-only matmul,
// backward.rs:118-120).  q, k, v, out are [batch*seq, heads*dh] row-major --
// head h of token (b, s) is the dh-slice starting at column h*dh -- so every
// per-(b,h) matrix is addressed in place through the GEMM's two batch levels
// (z = b*heads + h) with leading dimension heads*dh.  P holds the softmax
// probabilities [batch*heads, seq, seq] saved by the forward.
//
//   forward:   S = alpha * Q K^T,  P = softmax_rows(S),  O = P V
//   backward:  dV = P^T dO,  dP = dO V^T,  dS = P * (dP - rowsum(dP*P)),
//              dQ = alpha * dS K,  dK = alpha * dS^T Q
// with alpha = 1/sqrt(dh).  The forward is one kernel and the backward two, or
// one (attention_bf3.h), where bf3_fits or bf3_few; other shapes take the batched
// GEMMs and the one-wave-per-row softmax kernels.
#include <algorithm>
#include <cmath>

#include "attention_bf3.h"
#include "common.h"

namespace {

// Whether workgroups of 128 rows fill at least three quarters of the CUs.
bool fills(numrs_hip_ctx *ctx, int64_t S, int64_t Z) {
  return (S + 127) / 128 * Z * 4 >= 3 * std::max(ctx->num_cus, 1);
}

// Whether attention_bf3.h's kernels take the call: head sizes of whole 16-byte chunks up to 128; a
// staged block and four rows of P within 31-bit element offsets.
bool bf3_takes(int64_t S, int64_t Z, int64_t dh, int64_t li, int64_t lo) {
  return dh % 8 == 0 && dh <= 128 && Z < 65536 && S < (int64_t{1} << 28) && li < (int64_t{1} << 24) &&
         lo < (int64_t{1} << 24);
}

// And whether they are the faster ones.  Below 2^24 multiply-adds a product (the tiny GEMM's
// range), with fewer than 32 workgroups, or with heads above 64 on a part of the chip, the GEMMs
// and row kernels are as fast or faster: forward and backward on MI355X, B x S x H x dh,
// kernels | GEMMs: 2 x 256 x 4 x 64 43 | 57 us, 16 x 64 x 16 x 128 46 | 55, 1 x 1000 x 4 x 64 143 |
// 157; 1 x 1000 x 1 x 64 140 | 73, 4 x 256 x 8 x 128 92 | 76.
bool bf3_fits(numrs_hip_ctx *ctx, int64_t S, int64_t Z, int64_t dh, int64_t li, int64_t lo) {
  return bf3_takes(S, Z, dh, li, lo) && (double)Z * S * S * dh >= (double)(1 << 24) &&
         (S + 63) / 64 * Z >= 32 && (dh <= 64 || fills(ctx, S, Z));
}

// Heads up to 64 and at most one staged block of 128 rows, or whole ones up to `most`, a workgroup
// to a CU: one launch in place of three or six.  Forward, one head of 64 and eight, kernel | GEMMs:
// S = 64 8 | 10 and 9 | 11 us, 128 8 | 11 and 8 | 13, 256 12 | 14, 384 with four 17 | 26, 512 with
// two 21 | 30; but 192 13 | 12, 320 17 | 15.  Backward with the output: 64 11 | 13 and 12 | 14, 128
// 11 | 15 and 11 | 17, 256 17 | 19 and 18 | 30; but 192 17 | 15, 384 23 | 22, 512 29 | 24.
bool bf3_few(numrs_hip_ctx *ctx, int64_t S, int64_t Z, int64_t dh, int64_t li, int64_t lo, int64_t most) {
  return bf3_takes(S, Z, dh, li, lo) && dh <= 64 && (S + 63) / 64 * Z <= ctx->num_cus &&
         (S <= 128 || (S <= most && S % 128 == 0));
}

// Whether the backward with the output runs as one launch (attn::bwd_both_kernel): its workgroups
// of both kinds at most one to a CU.  Above that the two launches are as fast or faster: S = 384,
// 32 heads 42 us against 47, S = 512, 32 heads 55 against 61.
bool both_fit(numrs_hip_ctx *ctx, int64_t S, int64_t Z, int64_t dh) {
  return dh <= 64 && S <= attn::kMaxS && (S + 63) / 64 * Z * 2 <= ctx->num_cus && !fills(ctx, S, Z);
}

// Calls f with the configuration for head size dh and its grid: eight row groups of 16 where
// their workgroups fill the chip, else four (4 x 777 x 8 x 64: 193 us against 260; 1 x 1024 x 16 x
// 64: 238 against 159).
template <typename F>
void with_bf3(numrs_hip_ctx *ctx, int64_t S, int64_t Z, int64_t dh, F &&f) {
  auto go = [&](auto cfg) {
    using C = decltype(cfg);
    f(cfg, dim3((unsigned)((S + 16 * C::NW - 1) / (16 * C::NW)), (unsigned)Z));
  };
  if (!fills(ctx, S, Z)) {
    if (dh <= 32)
      go(attn::Cfg<32, 4, 2>{});
    else
      go(attn::Cfg<64, 4, 2>{});
  } else if (dh <= 32) {
    go(attn::Cfg<32, 8, 1>{});
  } else if (dh <= 64) {
    go(attn::Cfg<64, 8, 1>{});
  } else if (dh <= 96) {
    go(attn::Cfg<96, 8, 1>{});
  } else {
    go(attn::Cfg<128, 8, 1>{});
  }
}

// The backward kernels: D (from `out` where given) and dQ, then dV and dK, or all at once; any of
// the three may be null.
int bf3_backward(numrs_hip_ctx *ctx, const float *q, const float *k, const float *v, int64_t li, const float *P,
                 const float *out, const float *dout, int64_t lo, float *dq, float *dk, float *dv, int64_t B,
                 int64_t S, int64_t H, int64_t dh, int accumulate) {
  const float alpha = 1.0f / sqrtf((float)dh);
  const bool both = dq != nullptr && (dk != nullptr || dv != nullptr) && both_fit(ctx, S, B * H, dh);
  numrs_hip::TempBlock rows(ctx);  // D per query, from the first kernel to the second
  if (out == nullptr || !both)
    if (int rc = rows.alloc((size_t)(B * H * S) * sizeof(float))) return rc;
  float *D = rows.f();
  with_bf3(ctx, S, B * H, dh, [&](auto cfg, dim3 grid) {
    using C = decltype(cfg);
    const int l = (int)li, s = (int)S, h = (int)H, d = (int)dh;
    auto query = [&](auto mode, float *grad) {
      attn::bwd_query_kernel<C, decltype(mode)::value><<<grid, C::NT, 0, ctx->stream>>>(
          k, v, l, P, dout, out, lo, D, grad, s, h, d, alpha, accumulate);
    };
    const std::integral_constant<int, attn::kWalkD> walk;
    const std::integral_constant<int, attn::kOutD> from_out;
    if constexpr (C::NG > 1) {  // both_fit: only these
      auto together = [&](auto given) {
        attn::bwd_both_kernel<C, decltype(given)::value><<<dim3(2 * grid.x, grid.y), C::NT, 0, ctx->stream>>>(
            q, k, v, l, P, dout, out, (int)lo, D, dq, dk, dv, s, h, d, alpha, accumulate);
      };
      if (both && out != nullptr) return together(std::true_type{});
      if (both) {
        query(walk, nullptr);
        return together(std::false_type{});
      }
    }
    if (out != nullptr)
      query(from_out, dq);
    else
      query(walk, dq);
    if (dk != nullptr || dv != nullptr)
      attn::bwd_key_kernel<C><<<grid, C::NT, 0, ctx->stream>>>(q, v, l, P, dout, (int)lo, D, dk, dv, s, h, d, alpha,
                                                               accumulate);
  });
  return numrs_hip::check_launch(ctx, "attention backward");
}

int check(numrs_hip_ctx *ctx, int64_t B, int64_t S, int64_t H, int64_t D, int64_t ld_qkv,
          int64_t ld_out) {
  if (B <= 0 || S <= 0 || H <= 0 || D <= 0 || D % H != 0)
    return numrs_hip::fail(ctx, NUMRS_HIP_E_SHAPE,
                           "attention: batch, seq, heads > 0 and dim divisible by heads");
  if (ld_qkv < D || ld_out < D)
    return numrs_hip::fail(ctx, NUMRS_HIP_E_SHAPE, "attention: row strides below the dim");
  return NUMRS_HIP_OK;
}

}  // namespace

extern "C" {

// q, k, v rows (and dq, dk, dv in the backward) at stride ld_qkv, out / dout
// rows at stride ld_out: q, k, v may be column slices of one packed
// [B*S, 3D] projection (ld_qkv = 3D).
int numrs_hip_attention_forward_strided(numrs_hip_ctx *ctx, const float *q, const float *k,
                                        const float *v, int64_t ld_qkv, float *P, float *out,
                                        int64_t ld_out, int64_t B, int64_t S, int64_t H,
                                        int64_t D) {
  NRS_CHECK_CTX(ctx);
  if (int rc = check(ctx, B, S, H, D, ld_qkv, ld_out)) return rc;
  if (!q || !k || !v || !P || !out)
    return numrs_hip::fail(ctx, NUMRS_HIP_E_INVALID, "attention_forward: null pointer");
  const int64_t dh = D / H, Z = B * H, li = ld_qkv, lo = ld_out;
  const float alpha = 1.0f / sqrtf((float)dh);
  if (bf3_fits(ctx, S, Z, dh, li, lo) || bf3_few(ctx, S, Z, dh, li, lo, 512)) {
    const double a2 = (double)alpha * 1.4426950408889634;  // alpha log2 e
    const attn::Scale sc{(float)a2, (float)(a2 - (double)(float)a2)};
    with_bf3(ctx, S, Z, dh, [&](auto cfg, dim3 grid) {
      using C = decltype(cfg);
      auto go = [&](auto keep) {
        attn::fwd_kernel<C, decltype(keep)::value><<<grid, C::NT, 0, ctx->stream>>>(
            q, k, v, (int)li, P, out, lo, (int)S, (int)H, (int)dh, sc);
      };
      // all scores of a wave in registers: those of 256 keys, with the keys of a block halved
      // between two sets of waves of 512
      if (S <= 256) return go(std::integral_constant<int, 256 / C::BLK>{});
      if constexpr (C::NG > 1)
        if (S <= 512) return go(std::integral_constant<int, 512 / C::BLK>{});
      go(std::integral_constant<int, 0>{});
    });
    return numrs_hip::check_launch(ctx, "attn::fwd_kernel");
  }
  // S_z = alpha * Q_z K_z^T  -> P (row-major [S, S] per z)
  if (int rc = numrs_hip_gemm(ctx, q, li, k, li, P, S, S, dh, S, 0, 1, alpha, 0, Z, H, S * li, dh,
                              S * li, dh, H * S * S, S * S))
    return rc;
  // in-place row softmax (each row is read completely before it is written)
  if (int rc = numrs_hip_softmax_forward(ctx, P, P, Z * S, S, 1.0f)) return rc;
  // O_z = P_z V_z
  return numrs_hip_gemm(ctx, P, S, v, li, out, lo, S, S, dh, 0, 0, 1.0f, 0, Z, H, H * S * S,
                        S * S, S * li, dh, S * lo, dh);
}

int numrs_hip_attention_backward_strided(numrs_hip_ctx *ctx, const float *q, const float *k,
                                         const float *v, int64_t ld_qkv, const float *P,
                                         const float *dout, int64_t ld_out, float *dq, float *dk,
                                         float *dv, int64_t B, int64_t S, int64_t H, int64_t D,
                                         int accumulate) {
  NRS_CHECK_CTX(ctx);
  if (int rc = check(ctx, B, S, H, D, ld_qkv, ld_out)) return rc;
  if (!q || !k || !v || !P || !dout)
    return numrs_hip::fail(ctx, NUMRS_HIP_E_INVALID, "attention_backward: null input");
  const int64_t dh = D / H, Z = B * H, li = ld_qkv, lo = ld_out;
  const float alpha = 1.0f / sqrtf((float)dh);
  // dV_z = P_z^T dO_z
  auto dv_gemm = [&]() {
    return numrs_hip_gemm(ctx, P, S, dout, lo, dv, li, S, S, dh, 1, 0, 1.0f, accumulate, Z, H,
                          H * S * S, S * S, S * lo, dh, S * li, dh);
  };
  if (!dq && !dk) return dv ? dv_gemm() : NUMRS_HIP_OK;
  if (bf3_fits(ctx, S, Z, dh, li, lo))
    return bf3_backward(ctx, q, k, v, li, P, nullptr, dout, lo, dq, dk, dv, B, S, H, dh, accumulate);
  // dS lives in a block of its own: the products below may split their
  // reduction and write partials to the context workspace while reading dS.
  numrs_hip::TempBlock dSb(ctx);
  if (int rc = dSb.alloc((size_t)(Z * S * S) * sizeof(float))) return rc;
  float *dS = dSb.f();
  const numrs_hip::BatchedMat dSm{dS, S, H * S * S, S * S};
  const numrs_hip::BatchedMat Km{k, li, S * li, dh}, Qm{q, li, S * li, dh};
  const numrs_hip::BatchedOut dQ{dq, li, S * li, dh}, dK{dk, li, S * li, dh};
  if (dv)
    if (int rc = dv_gemm()) return rc;
  // dP_z = dO_z V_z^T
  if (int rc = numrs_hip_gemm(ctx, dout, lo, v, li, dS, S, S, dh, S, 0, 1, 1.0f, 0, Z, H, S * lo,
                              dh, S * li, dh, H * S * S, S * S))
    return rc;
  // dS = P * (dP - rowsum(dP * P)), in place over dP
  if (int rc = numrs_hip_softmax_backward(ctx, P, dS, dS, Z * S, S, 0)) return rc;
  // dQ_z = alpha * dS_z K_z ;  dK_z = alpha * dS_z^T Q_z  (one launch for both)
  return numrs_hip::gemm_nn_tn_pair(ctx, dSm, Km, dQ, Qm, dK, S, S, dh, alpha, accumulate, Z, H);
}

// The backward given also the forward's output `out` (rows at ld_out, like
// dout), from which the softmax backward's row totals come as dO . O.
int numrs_hip_attention_backward_out_strided(numrs_hip_ctx *ctx, const float *q, const float *k,
                                             const float *v, int64_t ld_qkv, const float *P,
                                             const float *out, const float *dout, int64_t ld_out,
                                             float *dq, float *dk, float *dv, int64_t B, int64_t S,
                                             int64_t H, int64_t D, int accumulate) {
  NRS_CHECK_CTX(ctx);
  if (int rc = check(ctx, B, S, H, D, ld_qkv, ld_out)) return rc;
  if (!q || !k || !v || !P || !dout || !out)
    return numrs_hip::fail(ctx, NUMRS_HIP_E_INVALID, "attention_backward: null input");
  const int64_t Z = B * H, dh = D / H;
  if ((dq || dk) && (bf3_fits(ctx, S, Z, dh, ld_qkv, ld_out) ||
                     (bf3_few(ctx, S, Z, dh, ld_qkv, ld_out, 256) && both_fit(ctx, S, Z, dh) && dq && (dk || dv))))
    return bf3_backward(ctx, q, k, v, ld_qkv, P, out, dout, ld_out, dq, dk, dv, B, S, H, D / H, accumulate);
  return numrs_hip_attention_backward_strided(ctx, q, k, v, ld_qkv, P, dout, ld_out, dq, dk, dv, B, S, H, D,
                                              accumulate);
}

int numrs_hip_attention_forward(numrs_hip_ctx *ctx, const float *q, const float *k, const float *v,
                                float *P, float *out, int64_t B, int64_t S, int64_t H,
                                int64_t D) {
  return numrs_hip_attention_forward_strided(ctx, q, k, v, D, P, out, D, B, S, H, D);
}

int numrs_hip_attention_backward(numrs_hip_ctx *ctx, const float *q, const float *k,
                                 const float *v, const float *P, const float *dout, float *dq,
                                 float *dk, float *dv, int64_t B, int64_t S, int64_t H, int64_t D,
                                 int accumulate) {
  return numrs_hip_attention_backward_strided(ctx, q, k, v, D, P, dout, D, dq, dk, dv, B, S, H, D,
                                              accumulate);
}

}  // extern "C"
