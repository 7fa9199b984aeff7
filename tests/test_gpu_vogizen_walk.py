"""A token of a Vogizen session by the launch that walks all layer runs (csrc/walk_vogizen.hip), against the single launches and the
plain statement of the equations: both element types and widths, loops, either mixer alone, shared key heads, taps, ranks, windows,
positions around the borders of its blocks of keys, a ring behind its end, its last position, and what follows it."""
import threading

import numpy as np
import pytest
import vogizen_gen as G
import vogizen_plain as P
from folder_helpers import BF16, F32, TOL, Opener, feed, generated_as_stepped, rel, tags_begin_anew, walks

pytestmark = pytest.mark.gpu


@pytest.fixture
def open_model(hip, tmp_path):
    o = Opener(hip, tmp_path, G)
    yield o
    o.close()


def model(width, kinds, loop=None, side=64, kv_heads=8, taps=4, q_rank=256, kv_rank=256, window=1024, vocab=200, **kw):
    d = G.delta(**{"heads": 16, "kv_heads": kv_heads, "dim": 128, "vdim": 128, "taps": taps, "ff": 3 * width, **kw.get("d", {})})
    a = G.latent(**{"heads": 16, "dim": 128, "vdim": 128, "q_rank": q_rank, "kv_rank": kv_rank, "window": window, "ff": 3 * width, **kw.get("a", {})})
    return G.config([d if k == "d" else a for k in kinds], width, vocab, side=side, loop=loop)


def three_ways(s, t, n, ref, dtype, what):
    """A pass of n tokens, seven tokens alone, a pass and a token behind them: walked twice, by single launches, and the plain ones."""
    got = []
    for on in (1, 1, 0):
        s.set_walks(on)
        s.reset()
        got.append(np.concatenate([s.step(t[:n], [n - 1]), feed(s, t[n : n + 7], [1]), feed(s, t[n + 7 : n + 13], [5, 1])]))
    assert np.array_equal(got[0], got[1]), what
    assert rel(got[0], got[2].astype(np.float64)) < TOL[dtype] / 2, what
    if ref is not None:
        assert rel(got[0], ref[n - 1 : n + 13]) < TOL[dtype], what
    return not np.array_equal(got[0][1:8], got[2][1:8])


@pytest.mark.parametrize("dtype", [F32, BF16])
@pytest.mark.parametrize("kw", [dict(width=1024, kinds="da", loop=(0, 2, 2), q_rank=768), dict(width=2048, kinds="da", loop=(1, 2, 2), side=128, q_rank=1024, kv_rank=512),
                                dict(width=1024, kinds="ad", side=128, kv_heads=16, taps=2, window=40), dict(width=2048, kinds="d", kv_heads=1, taps=3),
                                dict(width=1024, kinds="a", loop=(0, 1, 3), window=1)])
def test_walk_against_single_launches_and_plain(open_model, kw, dtype):
    cfg = model(**kw)
    s, w = open_model(cfg, None, dtype, 600)
    t = G.tokens(cfg, 300)
    ref, differ = P.forward(cfg, w, t), False
    for n in (1, 30, 62, 94, 126, 250):
        differ |= three_ways(s, t, n, ref, dtype, (kw, n))
    assert differ  # (the walk adds in another order: it was taken)


@pytest.mark.parametrize("dtype", [F32, BF16])
@pytest.mark.parametrize("kw,n", [(dict(width=1024, kinds="da", loop=(0, 2, 2)), 5), (dict(width=2048, kinds="da", loop=(1, 2, 2), side=128), 90),
                                  (dict(width=1024, kinds="ad", window=40), 60), (dict(width=2048, kinds="d"), 130)])
def test_generated_tokens(hip, open_model, kw, n, dtype):
    cfg = model(**kw)
    s, w = open_model(cfg, None, dtype, n + 20)
    generated_as_stepped(hip, s, G.tokens(cfg, n), 16, lambda t: P.forward(cfg, w, t), TOL[dtype])


def test_tags_begin_anew(hip, open_model):
    cfg = model(1024, "da", loop=(0, 2, 2))
    s, _ = open_model(cfg, None, BF16, 40)
    tags_begin_anew(hip, s, G.tokens(cfg, 14), 5)


@pytest.mark.parametrize("dtype", [F32, BF16])
def test_last_keys_and_a_ring(open_model, dtype):
    for kw, capacity, starts in ((dict(window=1024), 1100, (1017, 1050)), (dict(window=1100), 1200, (1018, 1060)), (dict(window=40), 2300, (2075, 2107, 2140)),
                                 (dict(window=1024), 3200, (3065, 3100))):
        cfg = model(1024, "ad", **kw)
        s, _ = open_model(cfg, None, dtype, capacity)
        t = G.tokens(cfg, capacity)
        for n in starts:
            assert three_ways(s, t, n, None, dtype, (kw, n)) or n > 1024  # (a window of 1100 is not the walk's from there on)


def test_shapes_the_walk_does_not_take(open_model):
    for kw in (dict(side=32), dict(taps=5), dict(taps=1), dict(d={"ff": 2048}), dict(a={"ff": None}), dict(q_rank=300), dict(d={"heads": 8}), dict(a={"vdim": 64}),
               dict(q_rank=1024), dict(width=1280)):
        cfg = model(**{"width": 1024, "kinds": "da", **kw})
        s, w = open_model(cfg, None, BF16, 40)
        t = G.tokens(cfg, 12)
        got = feed(s, t, [5, 1])
        s.set_walks(0)
        s.reset()
        assert np.array_equal(got, feed(s, t, [5, 1])), kw
        assert rel(got, P.forward(cfg, w, t)) < TOL[BF16], kw


@pytest.mark.parametrize("dtype", [F32, BF16])
def test_no_layers(open_model, dtype):
    cfg = G.config([], 1024, 90, loop=None)
    s, w = open_model(cfg, None, dtype, 20)
    t = G.tokens(cfg, 9)
    assert rel(feed(s, t, [4, 1]), P.forward(cfg, w, t)) < TOL[dtype]


@pytest.mark.parametrize("dtype", [F32, BF16])
def test_a_wait_that_is_given_up_leaves_the_single_launches(hip, open_model, dtype):
    cfg = model(1024, "da", loop=(0, 2, 2))
    s, _ = open_model(cfg, None, dtype, 120)
    t = G.tokens(cfg, 60)
    s.set_walks(0)
    single = feed(s, t, [40, 1])
    made = s.generate(t[:40], 30, [39, 50, 68])
    s.reset()
    s.set_walks(2)  # no vector crosses the chip that fast
    assert np.array_equal(feed(s, t[:41], [40, 1]), single[:41])
    assert walks(hip, s) == [1, 1]
    assert np.array_equal(feed(s, t[41:], [1]), single[41:])  # by single launches from then on
    assert walks(hip, s) == [1, 1]
    s.set_walks(2)
    again = s.generate(t[:40], 30, [39, 50, 68])
    assert walks(hip, s) == [30, 2]
    for k in ("tokens", "argmax", "dump"):
        assert np.array_equal(again[k], made[k]), k
    s.reset()
    s.set_walks(1)
    assert rel(feed(s, t, [40, 1]), single.astype(np.float64)) < TOL[dtype] / 2


def test_two_sessions_walk_on_two_threads(open_model):
    cfg = model(1024, "da", loop=(0, 2, 2))
    w = G.weights(cfg)
    sessions = [open_model(cfg, w, dtype, 300)[0] for dtype in (F32, BF16)]
    t = [G.tokens(cfg, 30 + 200 * k + 40, k) for k in range(2)]
    alone = [feed(s, x, [len(x) - 40, 1]) for s, x in zip(sessions, t)]
    got = [[], []]

    def run(k):
        for _ in range(6):
            sessions[k].reset()
            got[k].append(feed(sessions[k], t[k], [len(t[k]) - 40, 1]))

    threads = [threading.Thread(target=run, args=(k,)) for k in range(2)]
    for x in threads:
        x.start()
    for x in threads:
        x.join()
    for k in range(2):
        assert len(got[k]) == 6
        for g in got[k]:
            assert np.array_equal(g, alone[k])
