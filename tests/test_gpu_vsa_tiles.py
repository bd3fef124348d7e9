"""The tile choice of video sparse attention over many tiles: the edges of the
selection's forms (256 and 1024 tiles, and 64 and 8 of its and the coarse
branch's steps), and equal scores, of which the lower tiles win."""
import numpy as np
import pytest

import helpers as H
from test_gpu_vsa import TOL, _gpu_vsa

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tiles", [3, 63, 66, 255, 256, 257, 1023, 1024, 1026, 2050])
@pytest.mark.parametrize("tied", [False, True])
def test_many_tiles(gpu, oracle, tiles, tied):
    print("vsa %d tiles, tied %d" % (tiles, tied), flush=True)
    text, heads, hd = 70, 1, 64 if tiles % 2 else 128
    video = 4 * (tiles - 2) - 3  # two tiles of text; video tiles of four tokens in a row, the last of one
    n = text + video
    rng = np.random.default_rng(tiles)
    q, k, v, g = (rng.standard_normal((n, heads, hd)).astype(np.float32) for _ in range(4))
    if tied:
        q[:] = 0
    seq = (n, text, 0, video, 1, 1, video)
    o = _gpu_vsa(gpu, q, k, v, g, seq, 0.8)
    assert H.rel_fro(o, H.vsa_oracle(oracle, q, k, v, g, seq, 0.8)) <= TOL
