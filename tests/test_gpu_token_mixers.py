"""A token's attention takes its own key and value from where the launch makes them, its first block from loads that no
branch guards: every place of a block, the borders of the parts, and heads that fill none, some and all of a fragment."""
import numpy as np
import pytest
import ruvenex_gen as G
import ruvenex_plain as P
from folder_helpers import BF16, F32, TOL, Opener, feed, rel

pytestmark = pytest.mark.gpu


@pytest.fixture
def open_model(hip, tmp_path):
    o = Opener(hip, tmp_path, G)
    yield o
    o.close()


@pytest.mark.parametrize("dtype", [F32, BF16])
@pytest.mark.parametrize("dim,vdim,taps", [(2, 2, 1), (34, 18, 2), (64, 128, 3), (128, 40, 4), (126, 128, 4), (200, 256, 2)])
def test_every_place_of_a_block(open_model, dtype, dim, vdim, taps):
    cfg = G.config([G.layer_config(heads=3, kv_heads=1, dim=dim, vdim=vdim, taps=taps, rot_dims=dim // 4 * 2, rdim=dim, rvdim=vdim)], width=40)
    s, w = open_model(cfg, None, dtype, 300)
    t = G.tokens(cfg, 295)
    ref = P.forward(cfg, w, t)
    for sizes in ([1], [3, 1], [100, 1], [31, 98, 1]):  # (one token after another; the history carried over from passes)
        s.reset()
        got = feed(s, t, sizes)
        # bf16 keeps 8 bits of 24: the tolerance of the sessions' other tests; a key or value in a wrong place errs by its whole weight
        assert rel(got, ref) < TOL[dtype], (sizes, int(np.argmax(np.abs(got - ref).max(-1))))
