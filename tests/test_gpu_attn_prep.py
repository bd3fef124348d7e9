"""The attention preparation: several heads in one workgroup against one head
alone (the same bits), and rope dimensions that are no multiple of eight, which
take its channel-by-channel form, against the oracle."""
import numpy as np
import pytest

import test_gpu_attention as A

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,heads,hd,rot", [(300, 3, 128, 10), (65, 2, 64, 30), (130, 2, 128, 126), (64, 1, 64, 2),
                                            (127, 3, 64, 48), (200, 2, 128, 8)])
def test_rope_dims(gpu, oracle, n, heads, hd, rot):
    A.test_attention_qkv_branch(gpu, oracle, n, heads, hd, True, rot)
    A.test_attention_qkv_branch(gpu, oracle, n, heads, hd, False, rot)


# 64-slot tiles x heads: 34 x 121 (two heads to a workgroup, one left over),
# 32 x 195 (three, none left), 33 slots of 36 x 230 (four, two left)
@pytest.mark.parametrize("n,heads,hd", [(2111, 121, 64), (2048, 195, 64), (2100, 230, 128)])
def test_heads_together(gpu, n, heads, hd):
    F = gpu
    print("attention prep n=%d heads=%d hd=%d" % (n, heads, hd), flush=True)
    rng = np.random.default_rng(n + heads)
    inner, rot = heads * hd, 3 * hd // 4
    qkv = rng.standard_normal((n, 3 * inner), dtype=np.float32)
    qw, kw = (1 + 0.2 * rng.standard_normal((2, hd))).astype(np.float32)
    cos, sin = A._rope_tables(rng, n, rot)
    dn, dr = (A._buf(F, qw), A._buf(F, kw)), (A._buf(F, cos), A._buf(F, sin))

    def call(x, hs):
        do = F.DeviceBuffer(n * hs * hd * 4)
        F.attention_qkv_dev(A._buf(F, x), n, hs, hd, do, dn[0], dn[1], 1e-5, dr[0], dr[1], rot)
        F.synchronize()
        return do.download(np.float32, (n, hs, hd))

    got = call(qkv, heads)
    for h in (0, 1, 2, 3, heads // 2, heads - 2, heads - 1):
        one = np.concatenate([qkv[:, i * inner + h * hd:i * inner + (h + 1) * hd] for i in range(3)], 1)
        alone = call(np.ascontiguousarray(one), 1)[:, 0]
        assert np.array_equal(got[:, h].view(np.uint32), alone.view(np.uint32)), h
