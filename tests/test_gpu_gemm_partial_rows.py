"""The last tokens' partial blocks of k_gemm's 128-token tiles (16-byte stores of
the rows that exist) against the oracle, at the edges of its 32-token blocks, with
nothing stored past the last row; a y that is not 16-byte aligned takes the scalar
stores of the same tile and gives the same bits."""
import numpy as np
import pytest

import helpers as H

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [65, 95, 97, 127, 128, 257, 289, 383])
@pytest.mark.parametrize("N,epi", [(128, 0), (260, 0), (5120, 0), (384, 1), (256, 2)])
def test_partial_rows(gpu, oracle, M, N, epi):
    F = gpu
    K = 512  # too short to split: the tile itself stores y
    print("partial rows M=%d N=%d epi=%d" % (M, N, epi), flush=True)
    assert F.matmul_workspace_bytes(K, N, M, epi, prepared=True) == 0
    rng = np.random.default_rng(M + N)
    raw = F.synth_q4k_weights(M + N, 1, N, K, 0.05, 0.0)
    x = rng.standard_normal((M, K)).astype(np.float32)
    bias = rng.standard_normal(N).astype(np.float32)
    W = N // 2 if epi == 2 else N
    h, g = (rng.standard_normal((M, W)).astype(np.float32) for _ in range(2))
    dw, dx, db = (F.DeviceBuffer.from_array(a) for a in (raw, x, bias))
    dg = F.DeviceBuffer.from_array(np.concatenate([g.reshape(-1), np.zeros(4, np.float32)]))
    out = []
    for off in (0, 1):
        y0 = np.full(off + (M + 2) * W, 7, np.float32)
        if epi == 1:
            y0[off:off + M * W] = h.reshape(-1)
        dy = F.DeviceBuffer.from_array(y0)
        F.matmul_epi_dev(dw, K, N, dx, M, epi, dy.ptr + 4 * off, dg if epi == 1 else None, db)
        F.synchronize()
        y = dy.download(np.float32, y0.shape)
        assert (y[:off] == 7).all() and (y[off + M * W:] == 7).all()
        out.append(y[off:off + M * W].reshape(M, W))
    assert np.array_equal(out[0].view(np.uint32), out[1].view(np.uint32))
    ref = H.oracle_matmul(oracle, raw, K, N, x, bias)
    if epi == 1:
        ref = h + g * ref
    elif epi == 2:
        val, gate = ref[:, :W].astype(np.float64), ref[:, W:].astype(np.float64)
        ref = val * gate / (1 + np.exp(-gate))
    assert H.rel_fro(out[0], ref) <= 2e-3  # fp16 weights and activations, one rounding of 2^-11 each
