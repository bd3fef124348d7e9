"""The large products' two forms (k_gemm256 on weights decoded to fp16
fragments; k_gemm on the weights in place, which a call takes under capture)
give the same bits: an eager call against replays of the same call captured.
k_gemm itself is compared with the oracle in the tests of the GEMM path.

Shapes: the edges of the 256 x 256 tile in tokens and rows, output widths that
take the 16-byte stores, the scalar ones and both with a misaligned y, the
shortest K (one super-block: eight stages, two turns of the four-stage ring) and
one that is no multiple of the four super-blocks k_wfrag's workgroup decodes.
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


def _both(F, call, dy, y0):
    """The call run eagerly, then its captured form replayed twice (device-side fill between)."""
    dy.upload(y0)
    call()
    F.synchronize()
    eager = dy.download(np.float32, y0.shape)
    g = F.capture(call)
    try:
        for rep in range(2):
            dy.upload(y0)
            g.launch()
            F.synchronize()
            assert np.array_equal(eager.view(np.uint32), dy.download(np.float32, y0.shape).view(np.uint32)), rep
    finally:
        g.close()
    return eager


# tokens x rows chosen so that the tile counts take k_gemm256 by its rule; the
# last case is below it (both calls then run k_gemm)
CASES = [
    ("Q4_K", 4097, 256, 5001, 0, 0), ("Q4_K", 4097, 512, 5004, 0, 0), ("Q4_K", 4100, 768, 5120, 0, 4),
    ("Q4_K", 4095, 1280, 4993, 1, 0), ("Q4_K", 4096, 256, 5248, 1, 4), ("Q4_K", 4351, 512, 5248, 2, 0),
    ("Q4_K", 4097, 256, 5376, 2, 4), ("Q5_K", 4097, 512, 5001, 0, 0), ("Q5_K", 4352, 1280, 4992, 0, 0),
    ("Q6_K", 4097, 512, 5001, 0, 0), ("Q6_K", 4352, 1280, 4992, 0, 0), ("Q4_K", 1025, 256, 1001, 0, 0),
]


@pytest.mark.parametrize("name,M,K,N,epi,off", CASES)
def test_eager_equals_captured(gpu, name, M, K, N, epi, off):
    F = gpu
    print("gemm256 %s M=%d K=%d N=%d epi=%d offset %d" % (name, M, K, N, epi, off), flush=True)
    rng = np.random.default_rng(M + N)
    qt = H.QTYPES[name][0]
    x = rng.standard_normal((M, K)).astype(np.float32)
    W = N // 2 if epi == 2 else N
    dw, dx = F.DeviceBuffer.from_array(_weights(F, rng, name, N, K)), F.DeviceBuffer.from_array(x)
    db = F.DeviceBuffer.from_array(rng.standard_normal(N).astype(np.float32))
    extra = off // 4
    y0 = rng.standard_normal(M * W + extra).astype(np.float32)  # the gate residual adds to it
    dy = F.DeviceBuffer(y0.nbytes)
    dg = F.DeviceBuffer.from_array(rng.standard_normal(M * W + extra).astype(np.float32)) if epi == 1 else None

    def call():
        if epi == 0:
            F.matmul_dev(dw, K, N, dx, dy.ptr + off, M, db, qtype=qt)
        else:
            F.matmul_epi_dev(dw, K, N, dx, M, epi, dy.ptr + off, dg.ptr + off if dg else None, db)

    y = _both(F, call, dy, y0)
    assert np.isfinite(y).all() and np.array_equal(y[:extra], y0[:extra])
    for b in (dw, dx, db, dy, dg):
        if b is not None:
            b.close()


def test_streams_share_the_decoded_weights_safely(gpu):
    """Prepared products of different weights on two streams, back to back
    without a wait between: each result is the one its call gives alone."""
    F = gpu
    M, K, N = 4096, 512, 5120
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
