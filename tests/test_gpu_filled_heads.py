"""A token's attention where heads of 64 or 128 fill the kernel: its first positions, and the borders of one, two, up to four,
eight, sixteen and more parts of 128 keys, which are put together in different ways."""
import numpy as np
import pytest
import ruvenex_gen as G
import ruvenex_plain as P
import vogizen_gen
import vogizen_plain
from folder_helpers import BF16, F32, TOL, Opener, feed, feed_layers, rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [F32, BF16])
@pytest.mark.parametrize("heads,kv_heads,dim,taps", [(4, 2, 128, 4), (3, 1, 64, 4), (5, 1, 128, 1), (20, 1, 64, 1), (2, 2, 64, 2)])
def test_every_number_of_parts(hip, tmp_path, dtype, heads, kv_heads, dim, taps):
    cfg = G.config([G.layer_config(heads=heads, kv_heads=kv_heads, dim=dim, vdim=dim, taps=taps, rot_dims=dim // 2, rdim=8, rvdim=8)], width=40)
    o = Opener(hip, tmp_path, G)
    s, w = o(cfg, None, dtype, 2200)
    sizes, at = [1] * 6, 6
    for keys in (128, 256, 384, 512, 1024, 1152, 2048):  # single tokens across each
        sizes += [keys - 2 - at] + [1] * 4
        at = keys + 2
    t = G.tokens(cfg, at)
    ref = P.forward(cfg, w, t)
    got = feed(s, t, sizes)
    o.close()
    # the sessions' own tolerance: a part left out or weighed wrongly errs by its share of the weights, 1/17 and more
    assert rel(got, ref) < TOL[dtype], int(np.argmax(np.abs(got - ref).max(-1)))


@pytest.mark.parametrize("dtype", [F32, BF16])
@pytest.mark.parametrize("heads,kv_heads,dim,taps", [(4, 2, 128, 4), (3, 1, 64, 4), (5, 1, 128, 1), (20, 1, 64, 1)])
def test_bits_are_those_of_heads_of_any_size(hip, tmp_path, dtype, heads, kv_heads, dim, taps):
    """The same model with a tap of zeros more or less: 4 taps and 1 are the kernel that knows its sizes, 3 and 2 the one for any
    head.  A tap of zeros changes no sum, so all that can differ is how parts are put together."""
    def cfg(n):
        return G.config([G.layer_config(heads=heads, kv_heads=kv_heads, dim=dim, vdim=dim, taps=n, rot_dims=dim // 2, rdim=8, rvdim=8)], width=40)

    few, many = (3, 4) if taps == 4 else (1, 2)
    w = G.weights(cfg(few), 3)
    padded = {n: np.pad(a, ((0, 0), (1, 0))) if n.endswith(".conv") else a for n, a in w.items()}
    o = Opener(hip, tmp_path, G)
    s, s2 = o(cfg(few), w, dtype, 5000)[0], o(cfg(many), padded, dtype, 5000)[0]
    sizes, at = [1] * 6, 6
    for keys in (128, 256, 512, 640, 1024, 1152, 1700, 2048, 2176, 3072, 4096, 4900):  # from 512 on more parts than four
        sizes += [keys - 2 - at] + [1] * 4
        at = keys + 2
    t = G.tokens(cfg(few), at)
    a, b = feed(s, t, sizes), feed(s2, t, sizes)
    o.close()
    assert np.array_equal(a.view(np.uint32), b.view(np.uint32)), np.flatnonzero((a != b).any(-1))[:8]


@pytest.mark.parametrize("dtype", [F32, BF16])
@pytest.mark.parametrize("dim,window", [(128, 600), (64, 1000), (128, 1100), (64, 2000), (128, 2100)])
def test_parts_behind_a_window(hip, tmp_path, dtype, dim, window):
    """Five parts of 128 keys and more whose first key is not the sequence's: single tokens from the window's end on and where the
    cache's rows come round.  The attention alone, all else silenced: what the layer adds against the plain statement."""
    cfg = vogizen_gen.config([vogizen_gen.latent(heads=3, dim=dim, vdim=dim, window=window, scale=2 / dim**0.5, ff=None)], loop=None)
    w = vogizen_gen.weights(cfg, 5)
    w["l0.side.norm"] = np.zeros_like(w["l0.side.norm"])
    n = 2 * window + 40
    o = Opener(hip, tmp_path, vogizen_gen)
    s, _ = o(cfg, w, dtype, n)
    t = vogizen_gen.tokens(cfg, n)
    ref = []
    vogizen_plain.forward(cfg, w, t, layers_out=ref)
    half = window // 2
    got = feed_layers(s, t, [half, window - 2 - half] + [1] * 8 + [half, window - 50 - half] + [1] * 84)[0]
    o.close()
    x0 = vogizen_plain.embedding(cfg, w, np.asarray(t))
    at = np.r_[window - 2:window + 6, 2 * window - 44:n]
    assert rel((got - x0)[at], (ref[0] - x0)[at]) < TOL[dtype]
