"""The M > 32 MFMA GEMM at the edges of its rings and tiles: one block up to
past every weight group and stage of the 128-row kernel (groups of four, two
and one blocks, rings of three), K splits that start inside a group, ragged M
and N, in both tile heights (PBX_GEMM_M64=0 selects the 128-row tiles at any
size).  Every row within 1e-5 relative L2 of the oracle: the activations'
fp16 pair holds 2^-22 of a value and the sums are fp32 over at most 1536
terms (2^-24 times the square root of their number), ~1e-6 together."""
import numpy as np
import pytest

import oracle
import purebee_amd as pb
from tests.conftest import rel_l2
from tests.test_gpu_gemv import synth_matrix, weight_bytes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("t", [pb.TYPE_Q4_0, pb.TYPE_Q8_0, pb.TYPE_Q4_1, pb.TYPE_F16])
@pytest.mark.parametrize("blocks", [1, 2, 3, 4, 5, 8, 13, 48])
@pytest.mark.parametrize("M,N", [(40, 130), (129, 300)])
@pytest.mark.parametrize("tiles", [None, "0"])
def test_gemm_ring_edges(ctx, monkeypatch, t, blocks, M, N, tiles):
    if tiles is not None:
        monkeypatch.setenv("PBX_GEMM_M64", tiles)
    K = 32 * blocks
    print(f"[case] gemm type={t} M={M} N={N} K={K} tiles={tiles}", flush=True)
    raw = weight_bytes(t, synth_matrix(5 * N + K + M, N, K))
    X = pb.synth_normal(M + K, M * K).reshape(M, K)
    X[1] *= 1e-3
    X[2] *= 300.0
    w = ctx.upload(t, N, K, raw)
    Y = ctx.linear(w, X)
    w.free()
    for m in (0, 1, 2, 31, 32, M - 1):
        assert rel_l2(Y[m], oracle.matvec(t, X[m], raw, N, K)) <= 1e-5
    assert np.isfinite(Y).all()
