"""A token's attention where heads of 64 or 128 fill the kernel: its first positions, and the borders of one, two, up to four,
eight, sixteen and more parts of 128 keys, which are put together in different ways."""
import numpy as np
import pytest
import ruvenex_gen as G
import ruvenex_plain as P
from folder_helpers import BF16, F32, TOL, Opener, feed, rel

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
