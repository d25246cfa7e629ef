"""The one-launch GEMM for few activation rows (and every M of Q6_K): tile
edges in M and N, chunks of 8 blocks with a remainder, fewer chunks than
waves and more, the form that walks the tiles (tall N, K <= 2048).  Every row
within 1e-5 relative L2 of the oracle: activations keep 2^-22 of their row's
largest magnitude in a chunk, sums are fp32."""
import numpy as np
import pytest

import oracle
import purebee_amd as pb
from tests.conftest import rel_l2
from tests.test_gpu_gemv import synth_matrix, weight_bytes

pytestmark = pytest.mark.gpu

TYPES = [pb.TYPE_Q4_0, pb.TYPE_Q8_0, pb.TYPE_Q4_1, pb.TYPE_F16, pb.TYPE_Q6_K]


def raw_weights(t, seed, N, K):
    W = synth_matrix(seed, N, K)
    return oracle.quantize_q6_k(W) if t == pb.TYPE_Q6_K else weight_bytes(t, W)


def activations(M, K, seed):
    X = pb.synth_normal(seed, M * K).reshape(M, K)
    X[1] *= 1e-30
    X[2] *= 1e30
    X[3, : K // 2] *= 1e-4  # chunks of very different magnitude
    return X


def error(y, ref, x):
    """Relative L2 error; a few outputs can cancel to far less than the sums
    that they are made of (one output of row 0.02 * |x| typical size came out
    at 8e-4), whose rounding stays in proportion to |w| |x|, so the norm is
    taken as at least that of outputs without cancellation."""
    typical = 0.02 * np.linalg.norm(x.astype(np.float64)) * np.sqrt(len(ref))
    return np.linalg.norm(y.astype(np.float64) - ref) / max(np.linalg.norm(ref), typical)


def check(ctx, t, M, N, K, rows):
    print(f"[case] rows gemm type={t} M={M} N={N} K={K}", flush=True)
    raw = raw_weights(t, 3 * N + K + M, N, K)
    X = activations(M, K, M + N)
    bias = pb.synth_normal(3, N)
    w = ctx.upload(t, N, K, raw)
    Y, Yb = ctx.linear(w, X), ctx.linear(w, X, bias)
    w.free()
    for m in rows:
        ref = oracle.matvec(t, X[m], raw, N, K)
        assert error(Y[m], ref, X[m]) <= 1e-5
        if m not in (1, 2):  # the bias swamps or vanishes beside those rows
            assert error(Yb[m], ref + bias, X[m]) <= 1e-5


@pytest.mark.parametrize("t", TYPES)
@pytest.mark.parametrize("M", [4, 16, 17, 32])
@pytest.mark.parametrize("N,K", [(1, 256), (17, 512), (130, 2304), (3080, 256), (6200, 2560)])
def test_rows_tiles(ctx, t, M, N, K):
    check(ctx, t, M, N, K, [0, 1, 2, 3, M - 1])


@pytest.mark.parametrize("t", TYPES[:4])
@pytest.mark.parametrize("K", [32, 224, 288, 2080])
def test_rows_partial_chunks(ctx, t, K):
    check(ctx, t, 9, 50, K, [0, 1, 2, 3, 8])


@pytest.mark.parametrize("t", TYPES)
@pytest.mark.parametrize("M,N,K", [(5, 33000, 256), (20, 16500, 512)])
def test_rows_tile_loop(ctx, t, M, N, K):
    check(ctx, t, M, N, K, [0, 1, 2, 3, M - 1])


@pytest.mark.parametrize("M,N,K", [(33, 100, 256), (70, 300, 2304), (200, 2500, 512), (700, 48, 1024)])
def test_q6_k_many_rows(ctx, M, N, K):
    check(ctx, pb.TYPE_Q6_K, M, N, K, [0, 1, 2, 3, 31, 32, M - 1])


@pytest.mark.parametrize("t", TYPES)
def test_rows_non_finite_stays_in_its_row(ctx, t):
    M, N, K = 6, 40, 2304
    raw = raw_weights(t, 5, N, K)
    X = pb.synth_normal(8, M * K).reshape(M, K)
    X[2, 7] = np.inf
    X[4, 300] = np.nan
    w = ctx.upload(t, N, K, raw)
    Y = ctx.linear(w, X)
    w.free()
    assert not np.isfinite(Y[2]).any() and np.isnan(Y[4]).all()
    for m in (0, 1, 3, 5):
        assert rel_l2(Y[m], oracle.matvec(t, X[m], raw, N, K)) <= 1e-5


def test_q6_k_k_limit_is_refused(ctx):
    N, K = 2, 16640
    w = ctx.upload(pb.TYPE_Q6_K, N, K, raw_weights(pb.TYPE_Q6_K, 1, N, K))
    with pytest.raises(pb.PbxError):
        ctx.linear(w, np.zeros((4, K), np.float32))
    w.free()


@pytest.mark.parametrize("t", TYPES)
@pytest.mark.parametrize("M,K", [(6, 512), (40, 512), (130, 512), (40, 8448)])
def test_tiny_rows_stay_finite(ctx, t, M, K):
    """Rows whose largest magnitude lies below 2^-113, zeros among them: the
    power of two that scales a row stays finite.  N(0, 1) times 1e-36 with
    weights of 0.02: outputs around 1e-36, normal numbers; an activation keeps
    2^-22 of itself (its fp16 pair at the clamped scale still holds 20 bits of
    the row's largest magnitude), so 1e-5 as for the other rows.  K = 8448 is
    the preparation of rows too long for the registers."""
    N = 40
    print(f"[case] tiny rows type={t} M={M} N={N} K={K}", flush=True)
    raw = raw_weights(t, M + K, N, K)
    X = pb.synth_normal(M, M * K).reshape(M, K)
    X[1] *= 1e-36
    X[1, 5::3] = 0.0
    X[2] = 0.0
    w = ctx.upload(t, N, K, raw)
    Y = ctx.linear(w, X)
    w.free()
    assert np.isfinite(Y).all() and not Y[2].any()
    for m in (0, 1, M - 1):
        assert error(Y[m], oracle.matvec(t, X[m], raw, N, K), X[m]) <= 1e-5


@pytest.mark.parametrize("t", TYPES[:4])
@pytest.mark.parametrize("M,N,K", [(16, 1, 6144), (16, 70, 6176), (12, 2040, 8224), (9, 130, 12320),
                                   (8, 100, 8192), (5, 33, 20000), (16, 2048, 6144)])
def test_few_columns_long_rows(ctx, t, M, N, K):
    """K split over workgroups (pbx_gemm_<type>_p16): its tile edges in N, row
    counts short of the tile, K that the 8 splits and the steps of 8 blocks
    do not divide."""
    check(ctx, t, M, N, K, [0, 1, 2, 3, M - 1])


@pytest.mark.parametrize("t", TYPES[:4])
def test_many_columns_take_the_prepared_gemm(ctx, t):
    check(ctx, t, 32, 16390, 2592, [0, 1, 2, 3, 31])


@pytest.mark.parametrize("M,N,K", [(4, 48, 8192), (8, 1024, 2048), (16, 768, 2304), (100, 48, 1024),
                                   (8, 1025, 2048), (16, 770, 2304), (9, 911, 1024)])
def test_q6_k_both_sides_of_the_gemv_line(ctx, M, N, K):
    check(ctx, pb.TYPE_Q6_K, M, N, K, [0, 1, 2, 3, M - 1])


def test_q6_k_non_finite_rows_as_one_row(ctx):
    """An infinite or NaN activation gives a Q6_K output row the NaNs that the
    one-row GEMV gives it (every code is taken against an offset, so infinity
    meets infinity of the other sign), through the GEMM as well."""
    M, N, K = 6, 1400, 2048
    w = ctx.upload(pb.TYPE_Q6_K, N, K, raw_weights(pb.TYPE_Q6_K, 9, N, K))
    X = pb.synth_normal(10, M * K).reshape(M, K)
    X[1, 7], X[2, 300], X[4, 2047] = np.inf, -np.inf, np.nan
    Y = ctx.linear(w, X)
    for m in range(M):
        one = ctx.linear(w, X[m])
        assert np.array_equal(np.isnan(one), np.isnan(Y[m]))
        assert np.isnan(Y[m]).all() == (m in (1, 2, 4))
    w.free()


@pytest.mark.parametrize("t,M,N,K", [(pb.TYPE_Q4_0, 16, 70, 6176), (pb.TYPE_Q4_1, 7, 70, 8192),
                                     (pb.TYPE_Q8_0, 32, 16390, 2592), (pb.TYPE_Q6_K, 4, 48, 2048)])
def test_few_rows_noalloc_takes_the_same_kernels(ctx, t, M, N, K):
    w = ctx.upload(t, N, K, raw_weights(t, M, N, K))
    X = pb.synth_normal(N, M * K).reshape(M, K)
    dx, dy = ctx.alloc(M * K * 4).upload(X), [ctx.alloc(M * N * 4) for _ in range(2)]
    ctx.linear_dev(w, dx.ptr, M, dy[0].ptr)
    ctx.linear_dev_noalloc(w, dx.ptr, M, dy[1].ptr)
    ctx.sync()
    a, b = (d.download(np.float32, M * N) for d in dy)
    for d in (dx, *dy):
        d.free()
    w.free()
    assert np.isfinite(a).all() and np.array_equal(a, b)
