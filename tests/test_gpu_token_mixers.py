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


@pytest.mark.parametrize("dtype", [F32, BF16])
@pytest.mark.parametrize("width,ffs", [(33, [None]), (40, [7, None]), (130, [None, 300, 5]), (1030, [5000, 9, 2100])])
def test_weights_fetched_ahead(open_model, dtype, width, ffs):
    """The launch also reads weights of its layer's output and of the next layer's input: less and more than its budget,
    layers of different sizes, none behind the last."""
    cfg = G.config([G.layer_config(ff=ff) for ff in ffs], width=width)
    s, w = open_model(cfg, None, dtype, 40)
    t = G.tokens(cfg, 9)
    assert rel(feed(s, t, [1]), P.forward(cfg, w, t)) < TOL[dtype]  # nothing depends on what is read
