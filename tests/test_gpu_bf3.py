"""Products on the bf16 matrix cores (gemm_bf3.h) against float64: every tile shape at its
edges, odd sizes and addresses, split reductions, special values, and the mean error."""
import numpy as np
import pytest

from conftest import assert_contraction, rand
from numrs_amd import Context, StepGraph
from numrs_amd import _lib as L

pytestmark = pytest.mark.gpu


@pytest.fixture
def rng():
    return np.random.default_rng(97)


def _at(c, a, off):
    """`a` on the device `off` floats past a 16-byte boundary."""
    return c.to_device(np.concatenate([np.zeros(off, np.float32), a.ravel()])).view(off, a.shape)


def _product(c, A, B, ta, tb, off=0):
    M, N = A.shape[1 if ta else 0], B.shape[0 if tb else 1]
    C = c.to_device(np.full(M * N + off, 7.0, np.float32)).view(off, (M, N))
    c.matmul(_at(c, A, off), _at(c, B, off), C, trans_a=bool(ta), trans_b=bool(tb))
    return C.numpy()


# Tiles of 64 x 64 ((257, 33, 129): remainders of one row, column and step), with split
# reductions ((300, 1000, 70), (511, 1000, 513)), 128 x 64 (1001, 777, 1531), 128 x 128
# (2050, 300, 1030) and 256 x 128 ((2303, 97, 2177), (4097, 40, 1025); one row in the last
# tile: 4097 takes 256 x 128 only where rows are reduction-contiguous); K = 40 and 33 are two
# tiles, the first of 8 and of 1 steps; K = 32 and 64 whole tiles.
SIZES = [(257, 33, 129), (300, 1000, 70), (511, 1000, 513), (1001, 777, 1531), (2050, 300, 1030),
         (2303, 97, 2177), (4097, 40, 1025), (2048, 32, 2048), (1024, 64, 2048)]


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("M,K,N", SIZES)
def test_product(hip_ctx, rng, M, K, N, ta, tb):
    print(f"[gpu] bf3 product {M}x{K}x{N} ta={ta} tb={tb}", flush=True)
    A, B = rand(rng, (K, M) if ta else (M, K)), rand(rng, (N, K) if tb else (K, N))
    ref = (A.T if ta else A).astype(np.float64) @ (B.T if tb else B).astype(np.float64)
    for off in (0, 1):
        got = _product(hip_ctx, A, B, ta, tb, off)
        assert_contraction(got, ref, K, what=f"C at {off}")
        # fp32 sums of 32 steps (six roundings each at most) and of up to 32 such sums
        # between splits: well under sqrt(K / 32 + 6) units of 2^-24
        rel = np.linalg.norm(got - ref) / np.linalg.norm(ref)
        assert rel < np.sqrt(K / 32 + 6) * 2.0 ** -24, rel


@pytest.mark.parametrize("T,fin,fout", [(1000, 617, 1531), (4100, 510, 514), (1537, 65, 2049)])
def test_linear_pair(hip_ctx, rng, T, fin, fout):
    """The Linear backward's pair (NN with TN, bias sums) and matmul_backward's (NT with TN) in
    one grid, at odd sizes; accumulated into what is there."""
    print(f"[gpu] bf3 pair T={T} in={fin} out={fout}", flush=True)
    c, lib = hip_ctx, L.load()
    x, W, g = rand(rng, (T, fin)), rand(rng, (fout, fin)), rand(rng, (T, fout))
    x64, W64, g64 = (a.astype(np.float64) for a in (x, W, g))
    dx0, dw0 = rand(rng, (T, fin)), rand(rng, (fout, fin))
    xd, Wd, gd = (c.to_device(a) for a in (x, W, g))
    for acc in (0, 1):
        dx, dw, db = c.to_device(dx0), c.to_device(dw0), c.empty((fout,))
        assert lib.numrs_hip_linear_backward(c.handle, gd.ptr, xd.ptr, Wd.ptr, dx.ptr, dw.ptr,
                                             db.ptr, T, fin, fout, acc, acc, 0,
                                             L.UNBROADCAST_CORRECT) == 0
        assert_contraction(dx.numpy(), acc * dx0 + g64 @ W64, fout, what="dx")
        assert_contraction(dw.numpy(), acc * dw0 + g64.T @ x64, T, what="dW")
        assert_contraction(db.numpy(), g64.sum(0), T, what="db")
    dA, dB = c.empty((T, fin)), c.empty((fin, fout))
    Bd = c.to_device(np.ascontiguousarray(W.T))
    c.matmul_backward(gd, xd, Bd, dA, dB)
    assert_contraction(dA.numpy(), g64 @ W64, fout, what="dA")
    assert_contraction(dB.numpy(), x64.T @ g64, T, what="dB")


@pytest.mark.parametrize("T,fin,fout", [(300, 257, 300), (1000, 617, 1531), (8193, 130, 513),
                                        (4096, 512, 2048), (2100, 2050, 2305)])
@pytest.mark.parametrize("off,acc", [(0, 0), (1, 1)])
def test_bias_sums(hip_ctx, rng, T, fin, fout, off, acc):
    """A Linear's bias gradient, formed by the dW product's own tiles: every tile shape, odd last
    rows, split and whole reductions, accumulated, db at any address, values that are not finite."""
    print(f"[gpu] bf3 bias sums T={T} in={fin} out={fout} off={off} acc={acc}", flush=True)
    c, lib = hip_ctx, L.load()
    x, W, g, db0 = rand(rng, (T, fin)), rand(rng, (fout, fin)), rand(rng, (T, fout)), rand(rng, (fout,))
    xd, Wd, dx, dw = c.to_device(x), c.to_device(W), c.empty((T, fin)), c.empty((fout, fin))

    def run():
        db, gd = _at(c, db0, off), c.to_device(g)
        assert lib.numrs_hip_linear_backward(c.handle, gd.ptr, xd.ptr, Wd.ptr, dx.ptr, dw.ptr, db.ptr,
                                             T, fin, fout, 0, 0, acc, L.UNBROADCAST_CORRECT) == 0
        return db.numpy()

    got, ref = run(), acc * db0 + g.astype(np.float64).sum(0)
    # three roundings of eight steps, up to 16 tiles a partial sum, T / 512 of those, two of the
    # four threads', up to 32 splits' and db0's
    rel = np.linalg.norm(got - ref) / np.linalg.norm(ref)
    assert rel < np.sqrt(3 + 16 + T / 512 + 2 + 32 + 1) * 2.0 ** -24, rel
    assert np.array_equal(got, run())
    g[T - 1, 0], g[5, fout - 1], g[0, 7] = np.inf, np.nan, -np.inf
    bad = run()
    assert bad[0] == np.inf and np.isnan(bad[-1]) and bad[7] == -np.inf
    rest = np.setdiff1d(np.arange(fout), [0, 7, fout - 1])
    assert np.array_equal(bad[rest], got[rest])


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_special_values(hip_ctx, rng, ta, tb):
    """Infinities, NaN, magnitudes above bf16's largest, and rows that only they touch: the
    values that fp32 products and sums have."""
    M, K, N = 520, 200, 390
    A, B = rand(rng, (M, K)), rand(rng, (K, N))
    A[3, 7], A[100, 0], A[300, 199], A[519, 5] = np.inf, np.nan, -np.inf, 3.4e38
    A[400, :] = 1e-30
    A[401, :] = 0.0
    A[401, 9] = np.inf
    B[9, 0] = 0.0  # inf * 0
    B[11, 389] = np.inf
    B[5, 389] = 0.5  # 3.4e38 times more than 1 overflows in fp32, and inf - inf there is NaN
    got = _product(hip_ctx, np.ascontiguousarray(A.T) if ta else A,
                   np.ascontiguousarray(B.T) if tb else B, ta, tb)
    with np.errstate(all="ignore"):
        ref = A.astype(np.float64) @ B.astype(np.float64)
        ref = np.where(np.isfinite(ref) & (np.abs(ref) > np.finfo(np.float32).max),
                       np.copysign(np.inf, ref), ref)
    fine = np.isfinite(ref)
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    assert np.array_equal(got[np.isinf(ref)], ref[np.isinf(ref)])
    big = np.zeros(ref.shape, bool)
    big[519] = True  # sums around 3e38: relative only
    rest = fine & ~big
    assert_contraction(got[rest], ref[rest], K, what="finite")
    both = fine & big
    assert np.all(np.abs(got[both] - ref[both]) <= 1e-6 * np.abs(ref[both]))
    tiny = np.abs(got[400, fine[400]] - ref[400, fine[400]])
    assert tiny.max() <= 1e-6 * np.sqrt(K) * 1e-30


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("M,K,N", SIZES)
def test_special_values_of_every_shape(hip_ctx, rng, M, K, N, ta, tb):
    """A row, a column and their crossing that hold an infinity, a NaN or a value above 2^112,
    in the first and last blocks of every tile shape; every other output as without them."""
    print(f"[gpu] bf3 special values {M}x{K}x{N} ta={ta} tb={tb}", flush=True)
    A, B = rand(rng, (M, K)), rand(rng, (K, N))
    A[0, K - 1], A[M - 1, 0], A[M // 2, K // 2] = np.inf, 1e35, np.nan
    B[K // 3, N - 1], B[K - 1, 1] = -np.inf, 1e35
    got = _product(hip_ctx, np.ascontiguousarray(A.T) if ta else A,
                   np.ascontiguousarray(B.T) if tb else B, ta, tb)
    with np.errstate(all="ignore"):
        ref = A.astype(np.float64) @ B.astype(np.float64)
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    assert np.array_equal(got[np.isinf(ref)], ref[np.isinf(ref)])
    fine = np.isfinite(ref)
    large = np.zeros(ref.shape, bool)
    large[M - 1], large[:, 1] = True, True
    assert_contraction(got[fine & ~large], ref[fine & ~large], K, what="others")
    # sums of at most a few terms above the rest: rounded at their size
    rest = fine & large
    assert np.all(np.abs(got[rest] - ref[rest]) <= 1e-6 * np.abs(ref[rest]) + 1e-6 * 1e35)


@pytest.mark.parametrize("K", [64, 512, 2048])
def test_mean_error(hip_ctx, rng, K):
    """The matrix unit's sums round down; tiles of alternating sign cancel that.  Without them
    the mean error is -6e-9 of the rms; the mean of 2^22 errors of 1.5e-7 scatters by 7e-11."""
    M = N = 2048
    A, B = rand(rng, (M, K)), rand(rng, (N, K))
    ref = A.astype(np.float64) @ B.astype(np.float64).T
    got = _product(hip_ctx, A, B, 0, 1)
    assert abs((got - ref).mean()) / np.sqrt(np.mean(ref ** 2)) < 1e-9


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("a,b", [(1e-37, 1e10), (1e10, 3e-38), (1e-40, 1e30), (2e-36, 0.5), (1e-20, 1e-17),
                                 (1e20, 1e7), (1e30, 1e-36), (1e35, 1e-3)])
def test_small_and_large_operands(hip_ctx, rng, ta, tb, a, b):
    """Operands far from 1, down to fp32's subnormals and up to sums just under 2^96: the error
    relative to the result is that of ordinary operands (test_product).  Above 2^112 the fp32
    MFMAs' sums of 64 steps, twice that (measured for them: 1.9e-7)."""
    M, K, N = 520, 333, 390
    A, B = rand(rng, (M, K), a), rand(rng, (K, N), b)
    got = _product(hip_ctx, np.ascontiguousarray(A.T) if ta else A,
                   np.ascontiguousarray(B.T) if tb else B, ta, tb)
    ref = A.astype(np.float64) @ B.astype(np.float64)
    rel = np.linalg.norm(got - ref) / np.linalg.norm(ref)
    # results below 2^-126 are rounded to multiples of 2^-149
    least = np.sqrt(ref.size) * 2.0 ** -150 / np.linalg.norm(ref)
    assert rel < (2 if a > 1e33 else 1) * np.sqrt(K / 32 + 6) * 2.0 ** -24 + least, rel


def test_left_out_terms(hip_ctx):
    """Operands whose left-out products are the largest, 2^-24 of each product and of one sign:
    the result is off by that and no more."""
    M, K, N = 520, 256, 390
    x = np.float32(1 + 2.0 ** -8 - 2.0 ** -17)  # h = 1, m = 2^-8, l = -2^-17
    got = _product(hip_ctx, np.full((M, K), x), np.full((K, N), x), 0, 0)
    ref = K * float(x) ** 2
    assert np.abs(got / ref - 1).max() < (1.01 + np.sqrt(K / 32 + 6)) * 2.0 ** -24


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("batch,M,K,N", [(16, 256, 2048, 256), (3, 70, 5001, 333), (5, 64, 4100, 66)])
def test_batched_splits(hip_ctx, rng, batch, M, K, N, ta, tb):
    """Batched products of few tiles and a long reduction, cut into ranges: accumulated, at whole
    and odd sizes, the same bits in every call."""
    print(f"[gpu] bf3 batched splits {batch} x {M}x{K}x{N} ta={ta} tb={tb}", flush=True)
    c = hip_ctx
    A = rand(rng, (batch, K, M) if ta else (batch, M, K))
    B = rand(rng, (batch, N, K) if tb else (batch, K, N))
    C0 = rand(rng, (batch, M, N))
    Ad, Bd = c.to_device(A), c.to_device(B)
    got = []
    for _ in range(2):
        C = c.to_device(C0)
        c.matmul_batched(Ad, Bd, C, trans_a=bool(ta), trans_b=bool(tb), accumulate=True)
        got.append(C.numpy())
    a, b = A.astype(np.float64), B.astype(np.float64)
    ref = C0 + (a.transpose(0, 2, 1) if ta else a) @ (b.transpose(0, 2, 1) if tb else b)
    assert_contraction(got[0], ref, K, what="C")
    assert np.array_equal(*got)


@pytest.mark.parametrize("batch,M,K,N", [(4, 4096, 64, 64), (2, 5003, 130, 70), (3, 66, 64, 4100)])
def test_batched_pair_splits(hip_ctx, rng, batch, M, K, N):
    """matmul_backward over batches, one of the pair's products cut (M long: dB, N long: dA)."""
    print(f"[gpu] bf3 batched pair splits {batch} x {M}x{K}x{N}", flush=True)
    c = hip_ctx
    A, B, g = rand(rng, (batch, M, K)), rand(rng, (batch, K, N)), rand(rng, (batch, M, N))
    dA0, dB0 = rand(rng, A.shape), rand(rng, B.shape)
    dA, dB = c.to_device(dA0), c.to_device(dB0)
    c.matmul_backward_batched(c.to_device(g), c.to_device(A), c.to_device(B), dA, dB, accumulate=True)
    g64 = g.astype(np.float64)
    assert_contraction(dA.numpy(), dA0 + g64 @ B.astype(np.float64).transpose(0, 2, 1), N, what="dA")
    assert_contraction(dB.numpy(), dB0 + A.astype(np.float64).transpose(0, 2, 1) @ g64, M, what="dB")


@pytest.mark.parametrize("N", [24, 33])
def test_two_level_batch_splits(hip_ctx, rng, N):
    """Heads interleaved in B and C (two batch strides), the reduction cut; what lies between the
    heads' outputs stays."""
    b, H, M, K = 2, 3, 64, 3000
    print(f"[gpu] bf3 two-level batch splits N={N}", flush=True)
    c, lib = hip_ctx, L.load()
    A, B = rand(rng, (b * H, K, M)), rand(rng, (b, K, H + 1, N))
    C0 = rand(rng, (b, M, H + 1, N))
    Ad, Bd, C = c.to_device(A), c.to_device(B), c.to_device(C0)
    ld = (H + 1) * N
    assert lib.numrs_hip_gemm(c.handle, Ad.ptr, M, Bd.ptr, ld, C.ptr, ld, M, K, N, 1, 0, 0.5, 0, b * H, H,
                              H * K * M, K * M, K * ld, N, M * ld, N) == 0
    got = C.numpy()
    for z in range(b * H):
        ref = 0.5 * (A[z].astype(np.float64).T @ B[z // H, :, z % H].astype(np.float64))
        assert_contraction(got[z // H, :, z % H], ref, K, what=f"C[{z}]")
    assert np.array_equal(got[:, :, H], C0[:, :, H])


def test_batched_without_workspace(rng):
    """A recording must not grow the workspace: a batch that wants one runs unsplit there."""
    batch, M, K, N = 4, 128, 4096, 128
    A, B = rand(rng, (batch, M, K)), rand(rng, (batch, K, N))
    ref = A.astype(np.float64) @ B.astype(np.float64)
    with Context(0) as c:
        Ad, Bd, C, E = c.to_device(A), c.to_device(B), c.zeros((batch, M, N)), c.zeros((batch, M, N))
        graph = StepGraph(c, lambda: c.matmul_batched(Ad, Bd, C))
        try:
            for _ in range(3):
                C.fill(7.0)
                graph.replay()
                c.matmul_batched(Ad, Bd, E)  # eager: the workspace grows between the replays
                assert_contraction(C.numpy(), ref, K, what="replayed")
                assert_contraction(E.numpy(), ref, K, what="eager")
        finally:
            graph.close()
