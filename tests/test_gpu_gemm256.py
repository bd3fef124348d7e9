"""The large products' two forms (k_gemm256 on weights decoded to fp16
fragments; k_gemm on the weights in place, which a call takes under capture)
give the same bits: an eager call against replays of the same call captured.
k_gemm itself is compared with the oracle in the tests of the GEMM path.

Which of them ran shows in the free memory: the decoded weights are the only
thing an eager prepared product of this size allocates.

Shapes: the edges of the 256 x 256 tile in tokens and rows, output widths that
take the 16-byte stores, the scalar ones and both with a misaligned y, the
shortest K (one super-block: eight stages, two turns of the four-stage ring) and
ones that are no multiple of the four super-blocks k_wfrag's workgroup decodes;
activations of 2^-20 to 2^20 by the row, with outliers, a row of zeros, an infinity
and a NaN; short rows of whole tiles, which k_gemm takes.
"""
import ctypes

import numpy as np
import pytest

import helpers as H

pytestmark = pytest.mark.gpu


def _weights(F, rng, name, N, K):
    if name == "Q4_K":
        return F.synth_q4k_weights(N + K, 1, N, K, 0.05, 0.0)
    return H.random_blocks(rng, name, N, K, scale_lo=-12, scale_hi=-8)


def _free_bytes(F):
    """Free device memory, through the library's own HIP runtime."""
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert F.lib().hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def _fragment_bytes(K, N, epi):
    return ((N // 2 + 127) // 128 if epi == 2 else (N + 255) // 256) * 256 * K * 2


def _same(a, b):
    nan = np.isnan(a)
    return np.array_equal(nan, np.isnan(b)) and np.array_equal(a[~nan].view(np.uint32), b[~nan].view(np.uint32))


@pytest.fixture
def fresh(gpu):
    """The library without any workspace yet (shutdown frees it): a product that
    decodes its weights then takes their bytes from the free memory."""
    gpu.synchronize()
    gpu.shutdown()
    gpu.init(0)
    yield gpu
    gpu.synchronize()


def _both(F, call, dy, y0, decoded):
    """The call run eagerly, then its captured form replayed twice (device-side
    fill between); decoded: the bytes of decoded weights the eager call must take,
    or 0 if it must take none."""
    dy.upload(y0)
    F.synchronize()
    before = _free_bytes(F)
    call()
    F.synchronize()
    taken = before - _free_bytes(F)
    assert taken >= decoded if decoded else taken <= 0, (taken, decoded)
    eager = dy.download(np.float32, y0.shape)
    g = F.capture(call)
    try:
        for rep in range(2):
            dy.upload(y0)
            g.launch()
            F.synchronize()
            assert _same(eager, dy.download(np.float32, y0.shape)), rep
    finally:
        g.close()
    return eager


# (type, tokens, K, rows, epilogue, byte offset of y, whether the rule takes k_gemm256)
CASES = [
    ("Q4_K", 4097, 256, 5001, 0, 0, 1), ("Q4_K", 16384, 1792, 1004, 0, 0, 1), ("Q4_K", 16384, 1792, 1004, 0, 4, 1),
    ("Q4_K", 2561, 5120, 5120, 0, 0, 1), ("Q4_K", 4095, 1280, 4993, 1, 0, 1), ("Q4_K", 16384, 1792, 1004, 1, 0, 1),
    ("Q4_K", 16383, 1792, 1004, 1, 4, 1), ("Q4_K", 3016, 2816, 10752, 2, 0, 1), ("Q4_K", 4097, 3840, 10752, 2, 4, 1),
    ("Q5_K", 4097, 512, 5001, 0, 0, 1), ("Q5_K", 16384, 1280, 1000, 0, 0, 1), ("Q6_K", 4097, 512, 5001, 0, 0, 1),
    ("Q6_K", 16384, 1280, 1000, 0, 0, 1), ("Q4_K", 1025, 256, 1001, 0, 0, 0), ("Q4_K", 4096, 512, 5120, 0, 0, 0),
]


@pytest.mark.parametrize("name,M,K,N,epi,off,takes", CASES)
def test_eager_equals_captured(fresh, name, M, K, N, epi, off, takes):
    F = fresh
    print("gemm256 %s M=%d K=%d N=%d epi=%d offset %d" % (name, M, K, N, epi, off), flush=True)
    rng = np.random.default_rng(M + N)
    qt = H.QTYPES[name][0]
    x = rng.standard_normal((M, K), dtype=np.float32) * np.exp2(rng.integers(-20, 21, (M, 1))).astype(np.float32)
    x[rng.random((M, K)) < 0.01] *= 64
    x[5] = 0
    x[M - 1, K // 2] = np.inf
    x[M // 2, 0] = np.nan
    W = N // 2 if epi == 2 else N
    dw, dx = F.DeviceBuffer.from_array(_weights(F, rng, name, N, K)), F.DeviceBuffer.from_array(x)
    db = F.DeviceBuffer.from_array(rng.standard_normal(N).astype(np.float32))
    prep = F.DeviceBuffer(F.prepared_bytes(M, K))
    F.prepare_x_dev(dx, M, K, prep)
    extra = off // 4
    y0 = rng.standard_normal(M * W + extra, dtype=np.float32)  # the gate residual adds to it
    dy = F.DeviceBuffer(y0.nbytes)
    dg = F.DeviceBuffer.from_array(rng.standard_normal(M * W + extra, dtype=np.float32)) if epi == 1 else None

    def call():
        if epi == 0:
            F.matmul_prepared_dev(dw, K, N, prep, dy.ptr + off, M, db, qtype=qt)
        else:
            F.matmul_prepared_epi_dev(dw, K, N, prep, M, epi, dy.ptr + off, dg.ptr + off if dg else None, db)

    y = _both(F, call, dy, y0, _fragment_bytes(K, N, epi) if takes else 0)
    ok = np.isfinite(x).all(1)
    rows = y[extra:].reshape(M, W)
    assert np.isfinite(rows[ok]).all() and not np.isfinite(rows[~ok]).any() and np.array_equal(y[:extra], y0[:extra])
    for b in (dw, dx, db, prep, dy, dg):
        if b is not None:
            b.close()


def test_streams_share_the_decoded_weights_safely(gpu):
    """Prepared products of different weights on two streams, back to back
    without a wait between: each result is the one its call gives alone."""
    F = gpu
    M, K, N = 4096, 512, 5001
    print("gemm256 two streams M=%d K=%d N=%d" % (M, K, N), flush=True)
    rng = np.random.default_rng(5)
    x = rng.standard_normal((M, K)).astype(np.float32)
    dx, prep = F.DeviceBuffer.from_array(x), F.DeviceBuffer(F.prepared_bytes(M, K))
    F.prepare_x_dev(dx, M, K, prep)
    dws = [F.DeviceBuffer.from_array(F.synth_q4k_weights(i, 1, N, K, 0.05, 0.0)) for i in range(2)]
    dys = [F.DeviceBuffer(M * N * 4) for _ in range(2)]
    want = []
    for dw, dy in zip(dws, dys):
        F.matmul_prepared_dev(dw, K, N, prep, dy, M)
        F.synchronize()
        want.append(dy.download(np.uint32, (M, N)))
        dy.fill(0)
    F.synchronize()
    streams = [ctypes.c_void_p() for _ in range(2)]
    for s in streams:  # through the library's own HIP runtime; 1 = hipStreamNonBlocking
        assert F.lib().hipStreamCreateWithFlags(ctypes.byref(s), ctypes.c_uint(1)) == 0
    for _ in range(4):
        for s, dw, dy in zip(streams, dws, dys):
            F.matmul_prepared_dev(dw, K, N, prep, dy, M, stream_ptr=s)
    F.synchronize()
    for dy, w in zip(dys, want):
        assert np.array_equal(dy.download(np.uint32, (M, N)), w)
    for s in streams:
        assert F.lib().hipStreamDestroy(s) == 0


@pytest.fixture
def streams(fresh):
    """Three streams of the library's own HIP runtime; 1 = hipStreamNonBlocking."""
    made = [ctypes.c_void_p() for _ in range(3)]
    for s in made:
        assert fresh.lib().hipStreamCreateWithFlags(ctypes.byref(s), ctypes.c_uint(1)) == 0
    yield made
    fresh.synchronize()
    for s in made:
        assert fresh.lib().hipStreamDestroy(s) == 0


def test_streams_side_by_side(fresh, streams):
    """Prepared products of different weights and sizes on three streams, back to
    back without a wait between (two have decoded weights of their own, which
    grow while the others' products are at work, the third reads in place
    meanwhile): each result is the one its call gives alone."""
    F = fresh
    M = 4096
    shapes = [(512, 5001), (768, 5001), (1280, 5001)]
    print("gemm256 three streams M=%d" % M, flush=True)
    rng = np.random.default_rng(5)
    work = []
    for K, N in shapes:
        dx, prep = F.DeviceBuffer.from_array(rng.standard_normal((M, K), dtype=np.float32)), F.DeviceBuffer(F.prepared_bytes(M, K))
        F.prepare_x_dev(dx, M, K, prep)
        dw = F.DeviceBuffer.from_array(F.synth_q4k_weights(K, 1, N, K, 0.05, 0.0))
        work.append((K, N, dw, prep))
    F.synchronize()
    want = []
    for K, N, dw, prep in work:  # captured: read in place, nothing decoded before the streams run
        dy = F.DeviceBuffer(M * N * 4)
        g = F.capture(lambda: F.matmul_prepared_dev(dw, K, N, prep, dy, M))
        g.launch()
        F.synchronize()
        want.append(dy.download(np.uint32, (M, N)))
        g.close()
    before = _free_bytes(F)
    dys = [[F.DeviceBuffer(M * N * 4) for K, N in shapes] for _ in streams]
    ys = before - _free_bytes(F)
    for k in range(6):  # every stream runs every shape, small to large
        for i, s in enumerate(streams):
            K, N, dw, prep = work[(k // 2) % 3]
            F.matmul_prepared_dev(dw, K, N, prep, dys[i][(k // 2) % 3], M, stream_ptr=s)
    F.synchronize()
    assert before - _free_bytes(F) - ys >= _fragment_bytes(1280, 5001, 0), "no product decoded its weights"
    for per_stream in dys:
        for dy, w in zip(per_stream, want):
            assert np.array_equal(dy.download(np.uint32, w.shape), w)
