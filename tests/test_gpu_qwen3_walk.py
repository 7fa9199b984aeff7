"""Generated tokens of a Qwen3 session by the launch that walks all layers (csrc/walk_qwen3.hip), against the same session by
single launches and against the CPU loop: tokens, every step's argmax and two largest logits and the asked logits bit for bit,
where its branches change: heads that share their keys' scores (from 352 keys on), slices of values longer than what is loaded
ahead (from 769 keys on), the last position it takes (1279 keys), launches of up to four tokens."""
import ctypes as C
import threading

import numpy as np
import pytest
from folder_helpers import walk_tags_from, walks

pytestmark = pytest.mark.gpu

_SAME = ("tokens", "argmax", "top2", "dump")


def _model(rmi, tmp_path, name="m", **kw):
    path = str(tmp_path / (name + ".gguf"))
    rmi.gguf.write_synthetic_qwen3(path, seed=5, **{"n_layer": 2, "vocab": 3000, **kw})
    f = rmi.gguf.GGUFFile(path)
    return f.metadata, {k: t[2] for k, t in f.tensors.items()}


def _equal(a, b, what):
    for k in _SAME:
        assert np.array_equal(np.asarray(a[k]).view(np.uint32), np.asarray(b[k]).view(np.uint32)), (what, k)


@pytest.mark.parametrize("kw,drop,rounding", [
    ({}, (), "TIES_EVEN"), ({"n_head_kv": 16, "vocab": 2999}, (), "HALF_AWAY"), ({"n_head_kv": 2, "n_layer": 1, "vocab": 70}, (), "NEON"),
    ({"n_layer": 3}, ("attn_q_norm", "attn_k_norm"), "TIES_EVEN")])
def test_walk_is_the_single_launches_bit_for_bit(hip, tmp_path, kw, drop, rounding):
    meta, tensors = _model(hip, tmp_path, **kw)
    tensors = {n: t for n, t in tensors.items() if not any(d in n for d in drop)}
    s = hip.decode.Qwen3Session(meta, tensors, 1300, getattr(hip.hip, "ROUND_" + rounding))
    rng = np.random.default_rng(3)
    for n, new, passes in ((1, 20, 1), (2, 1, 1), (40, 17, 0), (62, 4, 1), (345, 16, 1), (762, 12, 1), (1262, 30, 1)):
        prompt = rng.integers(0, s.vocab, n, dtype=np.uint32)
        dumps = sorted({n - 1, n + new // 2 - 1, n + new - 2})
        s.set_prompt_passes(passes)
        s.set_walks(1)
        before = walks(hip, s)
        walked = s.generate(prompt, new, dumps)
        again = s.generate(prompt, new, dumps)
        after = walks(hip, s)
        assert (after[0] > before[0]) == (new > 1 or not passes) and after[1] == 0
        s.set_walks(0)
        single = s.generate(prompt, new, dumps)
        assert walks(hip, s) == after
        _equal(walked, single, (kw, n, new))
        _equal(again, single, (kw, n, new, "again"))
    s.close()


@pytest.mark.parametrize("width,heads,kv,ff", [(512, 8, 8, 1024), (512, 8, 1, 3072), (512, 16, 2, 2048), (512, 16, 16, 4096), (1024, 8, 4, 1024), (1024, 8, 8, 4096),
                                               (1024, 8, 2, 3072), (1024, 16, 4, 2048), (1024, 16, 8, 4096)])
def test_sizes_of_the_walk(hip, tmp_path, width, heads, kv, ff):
    meta, tensors = _model(hip, tmp_path, n_embd=width, n_head=heads, n_head_kv=kv, n_ff=ff, vocab=1500)
    s = hip.decode.Qwen3Session(meta, tensors, 1300)
    for n, new in ((1, 20), (345, 16), (764, 10), (1262, 24)):
        prompt = np.random.default_rng(n).integers(0, s.vocab, n, dtype=np.uint32)
        s.set_walks(1)
        before = walks(hip, s)
        walked = s.generate(prompt, new, [n - 1, n + new - 2])
        assert walks(hip, s)[0] > before[0] and walks(hip, s)[1] == 0
        s.set_walks(0)
        _equal(walked, s.generate(prompt, new, [n - 1, n + new - 2]), n)
    s.close()


@pytest.mark.parametrize("width,heads,kv,ff", [(768, 8, 4, 3072), (1024, 16, 8, 2560), (1024, 12, 4, 3072), (1024, 16, 8, 5120), (2048, 16, 8, 6144)])
def test_sizes_that_are_not_the_walks(hip, tmp_path, width, heads, kv, ff):
    meta, tensors = _model(hip, tmp_path, n_embd=width, n_head=heads, n_head_kv=kv, n_ff=ff, vocab=500, n_layer=1)
    s = hip.decode.Qwen3Session(meta, tensors, 60)
    assert s.generate(np.arange(30, dtype=np.uint32), 20)["tokens"].size == 20
    assert walks(hip, s) == [0, 0]
    s.close()


@pytest.mark.parametrize("n,new", [(1, 12), (348, 8), (766, 6)])
def test_walk_is_the_cpu_loop(hip, oracle, tmp_path, n, new):
    meta, tensors = _model(hip, tmp_path)
    pool = oracle.Pool(8)
    prompt = np.random.default_rng(n).integers(0, 3000, n, dtype=np.uint32)
    dumps = sorted({n - 1, n, n + new - 2})
    cpu = oracle.Qwen3Decoder(meta, tensors, pool).generate(prompt, new, dump_steps=dumps)
    s = hip.decode.Qwen3Session(meta, tensors, n + new)
    _equal(s.generate(prompt, new, dumps), cpu, n)
    assert walks(hip, s)[0] > 0 and walks(hip, s)[1] == 0
    s.close()
    pool.close()


def test_a_wait_that_is_given_up_leaves_the_single_launches(hip, tmp_path):
    meta, tensors = _model(hip, tmp_path)
    s = hip.decode.Qwen3Session(meta, tensors, 200)
    prompt = np.random.default_rng(8).integers(0, 3000, 100, dtype=np.uint32)
    good = s.generate(prompt, 40, [99, 120, 138])
    s.set_walks(2)  # no vector crosses the chip that fast
    assert walks(hip, s)[1] == 0
    _equal(s.generate(prompt, 40, [99, 120, 138]), good, "given up")
    given_up = walks(hip, s)
    assert given_up[1] == 1
    _equal(s.generate(prompt, 40, [99, 120, 138]), good, "single launches from then on")
    assert walks(hip, s) == given_up
    s.set_walks(1)
    _equal(s.generate(prompt, 40, [99, 120, 138]), good, "on again")
    assert walks(hip, s)[0] > given_up[0] and walks(hip, s)[1] == 1
    stop = int(good["tokens"][21])
    first = int(np.flatnonzero(good["tokens"] == stop)[0])
    s.set_stop_ids([stop])
    assert np.array_equal(s.generate(prompt, 40)["tokens"], good["tokens"][:first])
    s.close()


def test_tags_begin_anew(hip, tmp_path):
    """Four tokens a launch of two layers are 13 tags: launches across the last tag, with words of all tags before them."""
    meta, tensors = _model(hip, tmp_path)
    s = hip.decode.Qwen3Session(meta, tensors, 200)
    prompt = np.random.default_rng(9).integers(0, 3000, 20, dtype=np.uint32)
    want = s.generate(prompt, 70, [30, 60, 88])
    for left in (12, 13, 20, 40):
        walk_tags_from(hip, s, 2**32 - 1 - left)
        before = walks(hip, s)
        _equal(s.generate(prompt, 70, [30, 60, 88]), want, left)
        assert walks(hip, s)[0] > before[0] and walks(hip, s)[1] == 0
    s.close()


def test_largest_logits_of_every_wave(hip, tmp_path):
    """A tile of eight rows a wave (256 workgroups of eight), so the two largest logits lie in all roles' workgroups and in all of their waves.  A
    workgroup that merges all workgroups' largest logits keeps them apart from its own waves': those may not have been read yet."""
    meta, tensors = _model(hip, tmp_path, vocab=16384, n_layer=1)
    s = hip.decode.Qwen3Session(meta, tensors, 900)
    rng = np.random.default_rng(4)
    rows = []
    for n in (5, 300):
        prompt = rng.integers(0, s.vocab, n, dtype=np.uint32)
        s.set_prompt_passes(0)  # every position of the prompt by a walk, too: other tokens than the model's own
        s.set_walks(1)
        before = walks(hip, s)
        walked = s.generate(prompt, 300, [n + 298])
        assert walks(hip, s)[0] > before[0] and walks(hip, s)[1] == 0
        s.set_walks(0)
        _equal(walked, s.generate(prompt, 300, [n + 298]), n)
        rows.append(walked["argmax"])
    wave = np.concatenate(rows) // 8
    assert set(wave % 8) == set(range(8)) and ((wave // 8 >= 64) & (wave // 8 < 128)).any()
    s.close()


def test_a_session_walks_only_while_no_other_is_at_work(hip, tmp_path):
    meta, tensors = _model(hip, tmp_path)
    s = hip.decode.Qwen3Session(meta, tensors, 100)
    prompt = np.random.default_rng(7).integers(0, 3000, 30, dtype=np.uint32)
    alone, before = s.generate(prompt, 40, [60]), walks(hip, s)
    assert before[0] == 10  # 39 tokens by fours, and one launch ends at the logits asked for: other threads' work starts between them
    other = (C.c_uint8 * 8)()
    hip.hip.lib._ZN14RmiSessionBusyC1Ev(other)  # what another session's call holds
    try:
        _equal(s.generate(prompt, 40, [60]), alone, "beside another")
        assert walks(hip, s) == before
    finally:
        hip.hip.lib._ZN14RmiSessionBusyD1Ev(other)
    _equal(s.generate(prompt, 40, [60]), alone, "alone again")
    assert walks(hip, s)[0] == 2 * before[0]
    s.close()


def test_two_sessions_walk_on_two_threads(hip, tmp_path):
    meta, tensors = _model(hip, tmp_path)
    prompts = [np.random.default_rng(k).integers(0, 3000, 30 + 200 * k, dtype=np.uint32) for k in range(2)]
    sessions = [hip.decode.Qwen3Session(meta, tensors, 300) for _ in range(2)]
    alone = [s.generate(p, 40, [len(p) + 38]) for s, p in zip(sessions, prompts)]
    got = [[], []]

    def run(k):
        for _ in range(6):
            got[k].append(sessions[k].generate(prompts[k], 40, [len(prompts[k]) + 38]))

    threads = [threading.Thread(target=run, args=(k,)) for k in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for k in range(2):
        assert len(got[k]) == 6
        for g in got[k]:
            _equal(g, alone[k], k)
        assert walks(hip, sessions[k])[0] > 0 and walks(hip, sessions[k])[1] == 0
        sessions[k].close()
