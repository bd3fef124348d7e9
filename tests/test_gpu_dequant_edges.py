"""Decoding at the edges of a wavefront's 64 sixteen-value pieces: one block,
just under, at and over a wavefront and a workgroup, bit for bit against the
oracle, with nothing stored past the last value."""
import numpy as np
import pytest

import helpers as H

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name", ["Q8_0", "Q2_K", "Q3_K", "Q4_K", "Q5_K", "Q6_K"])
@pytest.mark.parametrize("pieces", [16, 48, 64, 80, 240, 256, 272, 1040])
def test_dequant_piece_counts(gpu, oracle, name, pieces):
    F = gpu
    print("dequant %s, %d pieces" % (name, pieces), flush=True)
    t = H.QTYPES[name][0]
    rows, cols = pieces // 16, 256
    raw = H.random_blocks(np.random.default_rng(pieces), name, rows, cols)
    src = F.DeviceBuffer.from_array(raw)
    dst = F.DeviceBuffer.from_array(np.full(rows * cols + 1024, 7, np.float32))
    F.dequant_dev(src, dst, rows, cols, qtype=t)
    F.synchronize()
    out = dst.download(np.float32, (rows * cols + 1024,))
    ref = H.oracle_dequant(oracle, raw, rows, cols, t)
    assert np.array_equal(out[:rows * cols].view(np.uint32), np.ascontiguousarray(ref).reshape(-1).view(np.uint32))
    assert (out[rows * cols:] == 7).all()
