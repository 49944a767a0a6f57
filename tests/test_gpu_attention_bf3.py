"""The attention kernels on the bf16 matrix cores (attention_bf3.h) against float64: ragged
sequences and head sizes, each of their configurations, partial and accumulated gradients, and
special values."""
import math

import numpy as np
import pytest

from conftest import assert_contraction, rand
from numrs_amd import _lib as L

pytestmark = pytest.mark.gpu

# Eight row groups (enough workgroups to fill the chip) or four; sequences below and above 256
# (scores kept or formed again; four row groups: 512); heads of 8 (padded to 32), 24, 40 and 64, 72
# (to 96) and 128; sequences one past, one short of and far from a block's end; 16 x 256 x 8 x 64 is
# the encoder block's.  Both kinds of the backward's workgroups in one launch (without the output
# after another for D): (2, 300, 16, 32), (2, 511, 8, 64) and (1, 512, 16, 64) (on all CUs) and the
# small ones; a launch each: (2, 300, 24, 32), (1, 513, 12, 64).  Below 2^24 multiply-adds one launch of few workgroups: (1, 1, 1, 8) to (4, 128, 4, 64), and (2, 128, 1,
# 64), (1, 256, 7, 64), (1, 512, 2, 64; its backward takes the GEMMs); all of them GEMMs: (1, 192, 2,
# 64), and heads of 96 on part of the chip.  (2, 200, 12, 32) and (8, 250, 20, 128): heads up to 32
# on part of the chip and of 128 on all of it, with the scores kept.
SHAPES = [(4, 130, 8, 40), (16, 129, 16, 8), (2, 300, 16, 32), (8, 257, 12, 72), (32, 100, 16, 24),
          (3, 520, 30, 128), (10, 255, 10, 96), (5, 321, 7, 64), (16, 256, 8, 64), (4, 383, 24, 64),
          (2, 300, 16, 96), (2, 511, 8, 64), (2, 300, 24, 32), (1, 1, 1, 8), (3, 5, 2, 16), (2, 64, 3, 64),
          (1, 65, 2, 40), (1, 127, 5, 64), (4, 128, 4, 64), (2, 128, 1, 64), (1, 256, 7, 64), (1, 512, 2, 64),
          (1, 512, 16, 64), (1, 513, 12, 64), (1, 384, 4, 56), (1, 192, 2, 64), (2, 200, 12, 32), (8, 250, 20, 128)]


def _ref(q, k, v, g, B, S, H):
    """P, out and the gradients in float64, [B, H, S, .] inside, q's layout outside."""
    dh = q.shape[1] // H
    split = lambda a: a.astype(np.float64).reshape(B, S, H, dh).transpose(0, 2, 1, 3)  # noqa: E731
    merge = lambda a: a.transpose(0, 2, 1, 3).reshape(B * S, H * dh)  # noqa: E731
    Q, K, V, G = (split(a) for a in (q, k, v, g))
    s = Q @ K.transpose(0, 1, 3, 2) / math.sqrt(dh)
    P = np.exp(s - s.max(-1, keepdims=True))
    P /= P.sum(-1, keepdims=True)
    dP = G @ V.transpose(0, 1, 3, 2)
    dS = P * (dP - (dP * P).sum(-1, keepdims=True)) / math.sqrt(dh)
    return (P.reshape(B * H, S, S), merge(P @ V), merge(dS @ K), merge(dS.transpose(0, 1, 3, 2) @ Q),
            merge(P.transpose(0, 1, 3, 2) @ G))


def _at(a, off):
    return a.ptr + 4 * off


@pytest.mark.parametrize("B,S,H,dh", SHAPES)
def test_forward_backward(hip_ctx, B, S, H, dh):
    print(f"[gpu] attention bf3 B={B} S={S} H={H} dh={dh}", flush=True)
    rng = np.random.default_rng(S * 131 + dh)
    D, c, lib = H * dh, hip_ctx, L.load()
    qkv, g, prev = rand(rng, (B * S, 3 * D)), rand(rng, (B * S, D)), rand(rng, (B * S, 3 * D))
    q, k, v = qkv[:, :D], qkv[:, D:2 * D], qkv[:, 2 * D:]
    P64, out64, *grads = _ref(q, k, v, g, B, S, H)
    ref = np.concatenate(grads, axis=1)
    x, gd = c.to_device(qkv), c.to_device(g)
    P, out = c.to_device(np.full((B * H, S, S), np.nan, np.float32)), c.empty((B * S, D))
    qp, kp, vp = x.ptr, _at(x, D), _at(x, 2 * D)
    assert lib.numrs_hip_attention_forward_strided(c.handle, qp, kp, vp, 3 * D, P.ptr, out.ptr, D,
                                                   B, S, H, D) == 0
    assert_contraction(P.numpy(), P64, dh, what="P")
    assert_contraction(out.numpy(), out64, S, what="out")
    for what, given, acc, keep in (("out", True, 0, (1, 1, 1)), ("no out", False, 0, (1, 1, 1)),
                                   ("acc", True, 1, (1, 1, 1)), ("dq", True, 0, (1, 0, 0)),
                                   ("dk", False, 1, (0, 1, 0)), ("dk dv", True, 0, (0, 1, 1))):
        d = c.to_device(prev)
        ptrs = [p if want else None for p, want in zip((d.ptr, _at(d, D), _at(d, 2 * D)), keep)]
        if given:
            rc = lib.numrs_hip_attention_backward_out_strided(
                c.handle, qp, kp, vp, 3 * D, P.ptr, out.ptr, gd.ptr, D, *ptrs, B, S, H, D, acc)
        else:
            rc = lib.numrs_hip_attention_backward_strided(
                c.handle, qp, kp, vp, 3 * D, P.ptr, gd.ptr, D, *ptrs, B, S, H, D, acc)
        assert rc == 0
        got = d.numpy()
        for i, want in enumerate(keep):
            sl = slice(i * D, (i + 1) * D)
            if want:
                assert_contraction(got[:, sl], acc * prev[:, sl] + ref[:, sl], S + dh,
                                   what=f"{what}: d{'qkv'[i]}")
            else:
                assert np.array_equal(got[:, sl], prev[:, sl]), f"{what}: d{'qkv'[i]} touched"


@pytest.mark.parametrize("B,S,H,dh", [(16, 200, 16, 64), (2, 300, 16, 64)])
def test_special_values(hip_ctx, B, S, H, dh):
    """An infinite key element (scores of +-inf: NaN rows, or probabilities of 0), an infinite
    value and magnitudes above bf16's largest: what fp32 products give."""
    rng = np.random.default_rng(5)
    D, c, lib = H * dh, hip_ctx, L.load()
    q, k, v, g = (rand(rng, (B * S, D)) for _ in range(4))
    k[7, 3] = np.inf         # head 0 of sequence 0: +inf or -inf scores by the sign of q[., 3]
    v[S + 9, dh + 1] = np.inf  # head 1 of sequence 1: its output column
    k[20, 2 * dh + 2] = 3.4e38
    q[20, 2 * dh + 2] = 0.0  # a score of 0 from it; the others overflow
    with np.errstate(all="ignore"):
        P64, out64, *_ = _ref(q, k, v, g, B, S, H)
    dev = [c.to_device(a) for a in (q, k, v)]
    P, out = c.empty((B * H, S, S)), c.empty((B * S, D))
    assert lib.numrs_hip_attention_forward(c.handle, *(a.ptr for a in dev), P.ptr, out.ptr, B, S, H, D) == 0
    p, o = P.numpy(), out.numpy()
    head = 2  # k = 3.4e38 times a q above 1 overflows in fp32 and not in float64
    ok = np.arange(B * H) != head
    assert np.array_equal(np.isnan(p[ok]), np.isnan(P64[ok]))
    assert_contraction(np.nan_to_num(p[ok]), np.nan_to_num(P64[ok]), dh, what="P")
    cols = np.ones((B * S, D), bool)
    cols[:S, head * dh:(head + 1) * dh] = False
    assert np.array_equal(np.isnan(o[cols]), np.isnan(out64[cols]))
    assert np.array_equal(np.isposinf(o[cols]), np.isposinf(out64[cols]))
    fine = cols & np.isfinite(out64)
    assert_contraction(o[fine], out64[fine], S, what="out")
    assert np.isfinite(p[head, 20]).all() and abs(p[head, 20].sum() - 1) < 1e-5


@pytest.mark.parametrize("B,S,H,dh", [(16, 200, 16, 64), (2, 300, 16, 64)])
def test_nan_keys(hip_ctx, B, S, H, dh):
    """NaN keys that fill one lane's four first keys, or a later group of four, or sit beside a
    finite one: every probability of the head's rows is NaN, and no other head's is."""
    rng = np.random.default_rng(6)
    D, c, lib = H * dh, hip_ctx, L.load()
    q, k, v = (rand(rng, (B * S, D)) for _ in range(3))
    heads = {0: slice(0, 4), 1: slice(4, 8), 2: slice(8, 12), 3: slice(12, 16), 4: slice(0, 16),
             5: slice(20, 24), 6: slice(2, 3), 7: slice(0, S), 8: slice(S - 1, S)}
    for h, rows in heads.items():
        k[rows, h * dh + 5] = np.nan
    k[S:S + 4, 5] = np.inf  # head 0 of sequence 1: scores of +inf or -inf, by the sign of q
    P, out = c.empty((B * H, S, S)), c.empty((B * S, D))
    dev = [c.to_device(a) for a in (q, k, v)]
    assert lib.numrs_hip_attention_forward(c.handle, *(a.ptr for a in dev), P.ptr, out.ptr, B, S, H, D) == 0
    p, o = P.numpy(), out.numpy()
    want = np.zeros(p.shape, bool)
    want[list(heads)] = True
    want[H] = (q[S:2 * S, 5] > 0)[:, None]  # inf - inf in those rows
    assert np.array_equal(np.isnan(p), want)
    assert np.array_equal(np.isnan(o.reshape(B, S, H, dh).transpose(0, 2, 1, 3)).reshape(B * H, S, dh),
                          np.broadcast_to(want[:, :, :1], (B * H, S, dh)))


@pytest.mark.parametrize("B,S,H,dh", [(16, 200, 16, 64), (2, 300, 16, 64)])
@pytest.mark.parametrize("given", [True, False])
def test_small_values(hip_ctx, B, S, H, dh, given):
    """Values, output gradients and probabilities near the end of fp32's range: the products
    have the relative error of ordinary ones (some 3e-7 of sums of 300 terms; the reference is
    formed of the probabilities that the forward left)."""
    rng = np.random.default_rng(8)
    D, c, lib = H * dh, hip_ctx, L.load()
    q, k = rand(rng, (B * S, D), 1e10), rand(rng, (B * S, D), 1e-10)
    v, g = rand(rng, (B * S, D)), rand(rng, (B * S, D), 1e-34)
    q[:, 0], k[:, 0] = 1e10, 0.0
    k[3::50, 0] = -6e-8  # head 0: scores of -75 at these keys, probabilities of 1e-35
    g[:, :dh] *= 1e30    # head 0: larger gradients
    split = lambda a: a.astype(np.float64).reshape(B, S, H, dh).transpose(0, 2, 1, 3)  # noqa: E731
    rel = lambda got, ref: np.linalg.norm(got - ref) / np.linalg.norm(ref)  # noqa: E731
    for scale in (1.0, 1e-37):
        vs = v * np.float32(scale)
        qd, kd, vd, gd = (c.to_device(a) for a in (q, k, vs, g))
        P, out, dq, dk, dv = c.empty((B * H, S, S)), *(c.empty((B * S, D)) for _ in range(4))
        assert lib.numrs_hip_attention_forward(c.handle, qd.ptr, kd.ptr, vd.ptr, P.ptr, out.ptr, B, S, H, D) == 0
        if given:
            rc = lib.numrs_hip_attention_backward_out_strided(
                c.handle, qd.ptr, kd.ptr, vd.ptr, D, P.ptr, out.ptr, gd.ptr, D, dq.ptr, dk.ptr, dv.ptr, B, S, H, D, 0)
        else:
            rc = lib.numrs_hip_attention_backward(c.handle, qd.ptr, kd.ptr, vd.ptr, P.ptr, gd.ptr, dq.ptr, dk.ptr,
                                                  dv.ptr, B, S, H, D, 0)
        assert rc == 0
        p = P.numpy().astype(np.float64).reshape(B, H, S, S)
        Q, V, G = split(q), split(vs), split(g)
        assert rel(split(out.numpy()), p @ V) < 1e-6
        dV, dV64 = split(dv.numpy()), p.transpose(0, 1, 3, 2) @ G
        few = np.isin((np.arange(B * S).reshape(B, S) - 3) % 50, 0)  # [B, S]
        for b in range(B):
            assert 0 < p[b, 0][:, few[b]].max() < 1e-33
            assert rel(dV[b, 0, few[b]], dV64[b, 0, few[b]]) < 1e-6
        assert rel(dV[:, 1:], dV64[:, 1:]) < 1e-6
        if scale == 1.0:  # else dO V^T is below fp32's range
            dP = G @ V.transpose(0, 1, 3, 2)
            dS = p * (dP - (dP * p).sum(-1, keepdims=True)) / math.sqrt(dh)
            # dP - D cancels: errors of 5e-7 of dP's size, not of the difference's
            assert rel(split(dk.numpy())[:, 1:], (dS.transpose(0, 1, 3, 2) @ Q)[:, 1:]) < 4e-6


def _same_kind(got, ref, what):
    """NaN and infinities where the reference has them, the rest within fp32's rounding of the
    head's largest value ([.., S, dh] arrays)."""
    assert np.array_equal(np.isnan(got), np.isnan(ref)), f"{what}: NaN"
    assert np.array_equal(got[np.isinf(ref)], ref[np.isinf(ref)]), f"{what}: inf"
    fine = np.isfinite(ref)
    top = np.abs(np.where(fine, ref, 0.0)).max(axis=(-2, -1), keepdims=True)
    err = np.abs(np.where(fine, got - np.where(fine, ref, 0.0), 0.0))
    assert np.all(err <= 2e-5 * top), f"{what}: {(err / np.maximum(top, 1e-300)).max()}"


# eight row groups of 16 and four (with the output in one launch, but for 2 x 400 x 20), heads of 8
# to 128
@pytest.mark.parametrize("B,S,H,dh", [(16, 200, 16, 64), (2, 300, 16, 64), (2, 200, 12, 32), (4, 383, 10, 64),
                                      (2, 400, 20, 48), (8, 257, 12, 72), (3, 520, 30, 128)])
@pytest.mark.parametrize("given", [True, False])
def test_backward_special_values(hip_ctx, B, S, H, dh, given):
    """Infinities, NaN and magnitudes of 2^112 and more in Q, K, V and dO: the gradients that
    fp32 arithmetic gives (float64 here, of the GPU's own P and output)."""
    print(f"[gpu] attention special values B={B} S={S} H={H} dh={dh} out={given}", flush=True)
    rng = np.random.default_rng(9)
    D, c, lib = H * dh, hip_ctx, L.load()
    q, k, v, g = (rand(rng, (B * S, D)) for _ in range(4))
    g[5, 3] = np.inf                        # head 0
    v[7, dh + 1] = np.inf                   # head 1
    q[9, 2 * dh + 2] = np.inf               # head 2
    g[11, 3 * dh], v[:S, 3 * dh] = 3.395e38, 1e-3 * v[:S, 3 * dh]
    k[20, 4 * dh + 2], q[:S, 4 * dh + 2] = 1e36, 0.0
    g[S - 1, 5 * dh + 4] = np.nan
    qd, kd, vd, gd = (c.to_device(a) for a in (q, k, v, g))
    P, out, dq, dk, dv = c.empty((B * H, S, S)), *(c.empty((B * S, D)) for _ in range(4))
    assert lib.numrs_hip_attention_forward(c.handle, qd.ptr, kd.ptr, vd.ptr, P.ptr, out.ptr, B, S, H, D) == 0
    if given:
        rc = lib.numrs_hip_attention_backward_out_strided(
            c.handle, qd.ptr, kd.ptr, vd.ptr, D, P.ptr, out.ptr, gd.ptr, D, dq.ptr, dk.ptr, dv.ptr, B, S, H, D, 0)
    else:
        rc = lib.numrs_hip_attention_backward(c.handle, qd.ptr, kd.ptr, vd.ptr, P.ptr, gd.ptr, dq.ptr, dk.ptr,
                                              dv.ptr, B, S, H, D, 0)
    assert rc == 0
    split = lambda a: a.astype(np.float64).reshape(B, S, H, dh).transpose(0, 2, 1, 3)  # noqa: E731
    Q, K, V, G, O = (split(a) for a in (q, k, v, g, out.numpy()))
    p = P.numpy().astype(np.float64).reshape(B, H, S, S)
    with np.errstate(all="ignore"):
        dP = G @ V.transpose(0, 1, 3, 2)
        total = (G * O).sum(-1, keepdims=True) if given else (p * dP).sum(-1, keepdims=True)
        dS = p * (dP - total)
        alpha = 1 / math.sqrt(dh)
        dK, dQ, dV = alpha * (dS.transpose(0, 1, 3, 2) @ Q), alpha * (dS @ K), p.transpose(0, 1, 3, 2) @ G
    _same_kind(split(dv.numpy()), dV, "dv")
    _same_kind(split(dq.numpy()), dQ, "dq")
    _same_kind(split(dk.numpy()), dK, "dk")


@pytest.mark.parametrize("B,S,H,dh", [(3, 5, 2, 16), (1, 127, 5, 64), (2, 128, 1, 40), (1, 256, 7, 64), (2, 300, 16, 32),
                                      (8, 257, 12, 72)])
def test_strides_and_addresses(hip_ctx, B, S, H, dh):
    """Rows at odd strides, every buffer one float past a 16-byte boundary, forward and backward
    with the output; what lies between the rows stays."""
    print(f"[gpu] attention bf3 strides B={B} S={S} H={H} dh={dh}", flush=True)
    rng = np.random.default_rng(S + dh)
    D, c, lib = H * dh, hip_ctx, L.load()
    li, lo, n = 3 * D + 5, D + 3, B * S
    x, g, o0, d0 = rand(rng, (n, li)), rand(rng, (n, lo)), rand(rng, (n, lo)), rand(rng, (n, li))
    q, k, v = x[:, :D], x[:, D:2 * D], x[:, 2 * D:3 * D]
    P64, out64, *grads = _ref(q, k, v, g[:, :D], B, S, H)

    def at(a):
        return c.to_device(np.concatenate([np.zeros(1, np.float32), a.ravel()])).view(1, a.shape)

    xd, gd, out, d = at(x), at(g), at(o0), at(d0)
    P = at(np.full((B * H, S, S), np.nan, np.float32))
    assert lib.numrs_hip_attention_forward_strided(c.handle, xd.ptr, _at(xd, D), _at(xd, 2 * D), li, P.ptr, out.ptr,
                                                   lo, B, S, H, D) == 0
    assert lib.numrs_hip_attention_backward_out_strided(
        c.handle, xd.ptr, _at(xd, D), _at(xd, 2 * D), li, P.ptr, out.ptr, gd.ptr, lo, d.ptr, _at(d, D), _at(d, 2 * D),
        B, S, H, D, 0) == 0
    assert_contraction(P.numpy(), P64, dh, what="P")
    got, gout = d.numpy(), out.numpy()
    assert_contraction(gout[:, :D], out64, S, what="out")
    assert_contraction(got[:, :3 * D], np.concatenate(grads, axis=1), S + dh, what="dq dk dv")
    assert np.array_equal(gout[:, D:], o0[:, D:]) and np.array_equal(got[:, 3 * D:], d0[:, 3 * D:])
