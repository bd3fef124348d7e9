"""Short F16 rows in one launch (k_short16) against the general route, which a
forced path still takes: the same bits, non-finite activations included, at the
edges of its 128 x 128 tiles and of its row lengths (8 to 128 by 8; 136 is past it)."""
import numpy as np
import pytest

import helpers as H

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,K,N,bias", [(1, 8, 1, True), (3, 96, 5376, True), (64, 32, 127, False),
                                        (65, 24, 129, True), (127, 128, 128, True), (128, 104, 257, False),
                                        (129, 96, 31, True), (300, 120, 1000, True), (2880, 96, 5376, True),
                                        (130, 136, 130, True)])
def test_short_rows_same_bits(gpu, M, K, N, bias):
    F = gpu
    print("short rows M=%d K=%d N=%d" % (M, K, N), flush=True)
    rng = np.random.default_rng(M + K + N)
    w = rng.standard_normal((N, K)).astype(np.float16)
    x = rng.standard_normal((M, K)).astype(np.float32) * np.exp2(rng.integers(-20, 20, (M, 1))).astype(np.float32)
    if M > 2:
        x[1] = 0
        x[2, K // 2] = np.inf
    if M > 64:
        x[M - 1, 0] = np.nan
    b = rng.standard_normal(N).astype(np.float32) if bias else None
    bufs = [F.DeviceBuffer.from_array(a) if a is not None else None for a in (w, x, b)]
    out = []
    for path in (F.PATH_AUTO, F.PATH_GEMM):
        y = F.DeviceBuffer.from_array(np.full((M + 1) * N, 7, np.float32))
        F.set_path(path)
        try:
            F.matmul_dev(bufs[0], K, N, bufs[1], y, M, bufs[2], qtype=F.FH3_QUANT_F16)
            F.synchronize()
        finally:
            F.set_path(F.PATH_AUTO)
        out.append(y.download(np.float32, (M + 1, N)))
    assert (out[0][M] == 7).all()
    nan = np.isnan(out[1])
    assert np.array_equal(np.isnan(out[0]), nan)
    assert np.array_equal(np.where(nan, 0, out[0]).view(np.uint32), np.where(nan, 0, out[1]).view(np.uint32))
    ok = np.isfinite(x).all(1)
    ref = x[ok].astype(np.float64) @ w.astype(np.float64).T + (0 if b is None else b)
    assert H.rel_fro(out[0][:M][ok], ref) <= 1e-3  # one rounding of x to fp16 (2^-11) and fp32 sums


@pytest.mark.parametrize("M", [1, 3, 16, 17, 33, 64, 65, 200])
@pytest.mark.parametrize("K", [8, 24, 32, 96, 104, 128])
def test_prepared_gives_the_same_bits(gpu, M, K):
    """The two-stage form, which runs k_skinny16 up to 64 tokens and k_gemm16
    above: rows of 2^-20 to 2^20, a row of zeros, an infinity, a NaN."""
    F = gpu
    N = 300
    print("short rows, prepared and direct M=%d K=%d" % (M, K), flush=True)
    rng = np.random.default_rng(M * 1000 + K)
    w = (rng.standard_normal((N, K)) * np.exp2(rng.integers(-8, 9, (N, K)))).astype(np.float16)
    x = (rng.standard_normal((M, K)) * np.exp2(rng.integers(-20, 21, (M, 1)))).astype(np.float32)
    if M > 3:
        x[1], x[2, K - 1], x[3, 0] = 0, np.inf, np.nan
    dw, dx, db = (F.DeviceBuffer.from_array(a) for a in (w, x, rng.standard_normal(N).astype(np.float32)))
    prep, dys = F.DeviceBuffer(F.prepared_bytes(M, K)), [F.DeviceBuffer(M * N * 4) for _ in range(2)]
    F.matmul_dev(dw, K, N, dx, dys[0], M, db, qtype=F.FH3_QUANT_F16)
    F.prepare_x_dev(dx, M, K, prep)
    F.matmul_prepared_dev(dw, K, N, prep, dys[1], M, db, qtype=F.FH3_QUANT_F16)
    F.synchronize()
    a, b = (d.download(np.float32, (M, N)) for d in dys)
    nan = np.isnan(a)
    assert np.array_equal(nan, np.isnan(b)) and np.array_equal(a[~nan].view(np.uint32), b[~nan].view(np.uint32))


@pytest.mark.parametrize("M,K,N,shift", [(300, 96, 96, 0), (257, 64, 128, 0), (1000, 128, 8, 0), (200, 96, 96, 4),
                                         (300, 32, 64, -1000)])
def test_output_over_the_activations(gpu, M, K, N, shift):
    """y at x (shift floats further): the result is the one two buffers give."""
    F = gpu
    print("y over x M=%d K=%d N=%d shift %d" % (M, K, N, shift), flush=True)
    rng = np.random.default_rng(M + N)
    w = rng.standard_normal((N, K)).astype(np.float16)
    x = rng.standard_normal((M, K)).astype(np.float32)
    dw, dx, dy = F.DeviceBuffer.from_array(w), F.DeviceBuffer.from_array(x), F.DeviceBuffer(M * N * 4)
    F.matmul_dev(dw, K, N, dx, dy, M, qtype=F.FH3_QUANT_F16)
    both = F.DeviceBuffer((2000 + M * max(K, N)) * 4)
    host = np.zeros(2000 + M * max(K, N), np.float32)
    host[1000:1000 + M * K] = x.reshape(-1)
    both.upload(host)
    F.matmul_dev(dw, K, N, both.ptr + 4000, both.ptr + 4 * (1000 + shift), M, qtype=F.FH3_QUANT_F16)
    F.synchronize()
    got = both.download(np.float32, host.shape)[1000 + shift:1000 + shift + M * N]
    assert np.array_equal(got.view(np.uint32), dy.download(np.uint32, (M * N,)))
