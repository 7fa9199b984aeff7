"""Products of one token whose rows take one, some and more rounds of a wave than are in flight, by few workgroups and by
many, with everything the epilogue may read (vectors, a table's row) or not."""
import numpy as np
import pytest
import ruvenex_gen as G
import ruvenex_plain as P
import vogizen_gen as VG
import vogizen_plain as VP
from folder_helpers import BF16, F32, TOL, Opener, feed, rel

pytestmark = pytest.mark.gpu


# width: 64 lanes of 16 bytes are 256 f32 or 512 bf16 elements a round; ff 9000: rows past 32 to a compute unit
@pytest.mark.parametrize("dtype", [F32, BF16])
@pytest.mark.parametrize("width,ff", [(256, 40), (516, 64), (1030, 513), (2052, 9000), (4104, 100)])
@pytest.mark.parametrize("gen,plain,layer", [(G, P, G.layer_config), (VG, VP, VG.latent)])
def test_rounds(hip, tmp_path, gen, plain, layer, dtype, width, ff):
    o = Opener(hip, tmp_path, gen)
    try:
        cfg = gen.config([layer(ff=ff)], width=width, vocab=50)
        s, w = o(cfg, None, dtype, 16)
        t = np.random.default_rng(1).integers(0, 50, 5)
        # f32 sums of n terms err by a few sqrt(n) 2^-24 of their size, far below the sessions' own tolerance; a piece
        # left out or added twice errs by about 1 / sqrt(n)
        assert rel(feed(s, t, [1]), plain.forward(cfg, w, t)) < TOL[dtype]
    finally:
        o.close()
