"""Video sparse attention with enough tiles and heads that the preparation takes
several heads to a workgroup (gathered slots and tile pooling included), the tile
scores 64 x 64 and the coarse branch eight query tiles at a time: every selected
head the bits it has alone, where all three take their other form."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# 66 tiles x heads: four heads to a workgroup, three left over; three, one left;
# two, one left.  rot 30 is no multiple of eight (the channel-by-channel rope).
@pytest.mark.parametrize("heads,hd,rot,gated", [(131, 64, 48, True), (131, 128, 96, False), (100, 128, 96, True),
                                                (67, 128, 30, True), (67, 64, 48, False)])
def test_heads_together(gpu, heads, hd, rot, gated):
    F = gpu
    print("vsa heads=%d hd=%d rot=%d gate=%d" % (heads, hd, rot, gated), flush=True)
    rng = np.random.default_rng(heads + hd)
    text, video = 70, 4 * 64 - 3  # two tiles of text; 64 video tiles of four tokens in a row, the last of one
    n, inner = text + video, heads * hd
    qkv = rng.standard_normal((n, 3 * inner), dtype=np.float32)
    gate = rng.standard_normal((n, inner), dtype=np.float32)
    qw, kw = (1 + 0.2 * rng.standard_normal((2, hd))).astype(np.float32)
    ang = rng.standard_normal((n, rot))
    bufs = [F.DeviceBuffer.from_array(a) for a in (qw, kw, np.cos(ang).astype(np.float32), np.sin(ang).astype(np.float32))]
    seq = F.seq_of(n, text, 0, video, grid=(1, 1, video))

    def call(x, g, hs):
        dx, dg, do = F.DeviceBuffer.from_array(x), F.DeviceBuffer.from_array(g), F.DeviceBuffer(n * hs * hd * 4)
        F.vsa_attention_qkv_dev(dx, dg if gated else None, do, seq, hs, hd, 0.8, 64, bufs[0], bufs[1], 1e-5, bufs[2],
                                bufs[3], rot)
        F.synchronize()
        return do.download(np.float32, (n, hs, hd))

    got = call(qkv, gate, heads)
    assert np.isfinite(got).all()
    for h in (0, 1, 2, 3, 4, heads // 2, heads - 3, heads - 2, heads - 1):
        one = np.concatenate([qkv[:, i * inner + h * hd:i * inner + (h + 1) * hd] for i in range(3)], 1)
        alone = call(one, np.ascontiguousarray(gate[:, h * hd:(h + 1) * hd]), 1)[:, 0]
        assert np.array_equal(got[:, h].view(np.uint32), alone.view(np.uint32)), h
