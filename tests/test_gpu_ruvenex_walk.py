"""A token of a Ruvenex session by the launch that walks all layers (csrc/walk_ruvenex.hip), against the single launches and the
plain statement of the equations: heads that share keys, taps, rotations and feed-forwards at the edges of what it takes, positions
around the borders of its blocks of keys, its first and last position, and what follows it."""
import threading

import numpy as np
import pytest
import ruvenex_gen as G
import ruvenex_plain as P
from folder_helpers import BF16, F32, TOL, Opener, feed, generated_as_stepped, rel, tags_begin_anew, walks

pytestmark = pytest.mark.gpu


@pytest.fixture
def open_model(hip, tmp_path):
    o = Opener(hip, tmp_path, G)
    yield o
    o.close()


def model(n_layer=2, vocab=300, **kw):
    return G.config([G.layer_config(**{"dim": 128, "vdim": 128, "rdim": 128, "rvdim": 128, **kw})] * n_layer, 1024, vocab)


SHAPES = [dict(heads=4, kv_heads=2, taps=4, rot_dims=64, rheads=2, ff=512),
          dict(heads=8, kv_heads=1, taps=2, rot_dims=0, rheads=4, ff=250, n_layer=3),
          dict(heads=2, kv_heads=2, taps=3, rot_dims=128, rheads=2, ff=256, vocab=77, left_scale=-1.5, right_scale=0.3),
          dict(heads=16, kv_heads=8, taps=4, rot_dims=64, rheads=8, ff=3072)]


@pytest.mark.parametrize("kw", SHAPES)
def test_walk_against_single_launches_and_plain(open_model, kw):
    cfg = model(**kw)
    s, w = open_model(cfg, None, BF16, 530)
    t = G.tokens(cfg, 530)
    ref, differ = P.forward(cfg, w, t), False
    for n in (1, 29, 62, 94, 126, 254, 382, 508):  # then single tokens at n .. n + 6, across a border
        got = {}
        for on in (1, 0):
            s.set_walks(on)
            s.reset()
            first = s.step(t[:n], [n - 1])
            steps = feed(s, t[n : n + 7], [1])
            after = feed(s, t[n + 7 : n + 13], [5, 1])  # a pass and a token behind what the walk left
            got[on] = np.concatenate([first, steps, after])
        assert rel(got[1], ref[n - 1 : n + 13]) < TOL[BF16], n
        assert rel(got[1], got[0].astype(np.float64)) < TOL[BF16] / 2, n
        assert np.array_equal(got[1][0], got[0][0])  # a pass is a pass
        differ |= not np.array_equal(got[1], got[0])
    assert differ  # (the walk adds in another order: it was taken, though most logits come from the same bf16 values)


@pytest.mark.parametrize("kw,n", [(SHAPES[0], 5), (SHAPES[1], 120), (SHAPES[2], 250), (SHAPES[3], 40)])
def test_generated_tokens(hip, open_model, kw, n):
    cfg = model(**kw)
    s, w = open_model(cfg, None, BF16, n + 20)
    generated_as_stepped(hip, s, G.tokens(cfg, n), 16, lambda t: P.forward(cfg, w, t), TOL[BF16])


def test_tags_begin_anew(hip, open_model):
    cfg = model(**SHAPES[0], n_layer=3)
    s, _ = open_model(cfg, None, BF16, 40)
    tags_begin_anew(hip, s, G.tokens(cfg, 14), 4)


def test_shapes_the_walk_does_not_take(open_model):
    for kw in (dict(ff=None), dict(heads=3, kv_heads=1), dict(taps=1), dict(taps=5), dict(ff=300), dict(vdim=64), dict(rheads=3),
               dict(heads=16, kv_heads=8, rheads=16, ff=3072)):  # (the last: more workgroups than compute units)
        cfg = model(**{"heads": 2, "kv_heads": 1, "ff": 256, **kw})
        s, w = open_model(cfg, None, BF16, 40)
        t = G.tokens(cfg, 12)
        got = feed(s, t, [5, 1])
        s.set_walks(0)
        s.reset()
        assert np.array_equal(got, feed(s, t, [5, 1])), kw
        assert rel(got, P.forward(cfg, w, t)) < TOL[BF16], kw


def test_one_layer_goes_by_single_launches(open_model):
    """Its walk would write the stream where workgroups that have not started yet read the embedding."""
    cfg = model(**SHAPES[0], n_layer=1)
    s, w = open_model(cfg, None, BF16, 80)
    t = G.tokens(cfg, 60)
    assert rel(feed(s, t, [40, 1]), P.forward(cfg, w, t)) < TOL[BF16]
    got = []
    for on in (1, 0):
        s.set_walks(on)
        s.reset()
        got.append((feed(s, t, [40, 1]), s.generate(t[:40], 30, [39, 50, 68])))
    assert np.array_equal(got[0][0], got[1][0])
    for k in ("tokens", "argmax", "dump"):
        assert np.array_equal(got[0][1][k], got[1][1][k]), k


def test_no_layers(open_model):
    cfg = G.config([], 1024, 90)
    for dtype in (BF16, F32):
        s, w = open_model(cfg, None, dtype, 20)
        t = G.tokens(cfg, 9)
        assert rel(feed(s, t, [4, 1]), P.forward(cfg, w, t)) < TOL[dtype]


def test_a_wait_that_is_given_up_leaves_the_single_launches(hip, open_model):
    cfg = model(**SHAPES[0])
    s, _ = open_model(cfg, None, BF16, 120)
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
    assert rel(feed(s, t, [40, 1]), single.astype(np.float64)) < TOL[BF16] / 2


def test_two_sessions_walk_on_two_threads(open_model):
    cfg = model(**SHAPES[0])
    w = G.weights(cfg)
    sessions = [open_model(cfg, w, BF16, 300)[0] for _ in range(2)]
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
