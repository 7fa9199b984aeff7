"""What the GPU tests of the sessions share."""
import ctypes as C

import numpy as np

F32, BF16 = "float32", "bfloat16"
TOL = {F32: 3e-5, BF16: 4e-2}


def rel(got, want):
    """Largest row error: root mean square over the row's, against the typical row's size."""
    d = np.asarray(got, np.float64) - want
    return float(np.sqrt((d * d).mean(-1)).max() / np.sqrt((want * want).mean()))


def portions(n, sizes):
    """Slices that cut n tokens into portions of the given sizes (the last one repeats)."""
    out, at = [], 0
    while at < n:
        k = min(sizes[min(len(out), len(sizes) - 1)], n - at)
        out.append(slice(at, at + k))
        at += k
    return out


def feed(s, tokens, sizes):
    """Logits of every position, the tokens cut into portions."""
    return np.concatenate([s.step(tokens[p], range(p.stop - p.start)) for p in portions(len(tokens), sizes)])


def feed_layers(s, tokens, sizes):
    """The residual stream behind every layer run, the tokens cut into portions."""
    return np.concatenate([s.step(tokens[p], (), layers=True)[1] for p in portions(len(tokens), sizes)], 1)


def walks(hip, s):
    """[walks enqueued, sequences or tokens whose walk was given up] of a session so far, by the library's own function (csrc/session.h)."""
    counts = (C.c_uint64 * 2)()
    hip.hip.lib._Z23rmi_session_walk_countsPK10RmiSessionPm(C.c_void_p(s._h if isinstance(s._h, int) else s._h.value), counts)
    return list(counts)


def walk_tags_from(hip, s, tag0):
    """The session's next walk takes the tags behind tag0: all words of earlier ones have to be below."""
    hip.hip.lib._Z26rmi_session_walk_tags_fromP10RmiSessionj(C.c_void_p(s._h if isinstance(s._h, int) else s._h.value), C.c_uint32(tag0))


def generated_as_stepped(hip, s, prompt, new, ref, tol):
    """A generation whose tokens are walked, its embeddings by the launches that sample: the bits of the same tokens by steps, whose walks embed
    them, tokens that are the logits' largest, and logits within tol of ref(tokens) (by single launches within half of it)."""
    n = len(prompt)
    s.set_walks(1)
    before = walks(hip, s)
    made = s.generate(prompt, new, range(n - 1, n + new - 1))
    assert walks(hip, s) == [before[0] + new - 1, before[1]]
    tokens = [*prompt, *made["tokens"].tolist()]
    assert np.array_equal(made["tokens"], made["dump"].argmax(-1)) and np.array_equal(made["tokens"], made["argmax"][n - 1 :])
    assert np.array_equal(made["top2"][n - 1 :], -np.sort(-made["dump"], -1)[:, :2])
    want = ref(tokens[:-1])[n - 1 :]
    assert rel(made["dump"], want) < tol
    for on in (1, 0):
        s.set_walks(on)
        s.reset()
        before = walks(hip, s)
        stepped = np.concatenate([s.step(prompt, [n - 1]), feed(s, tokens[n:-1], [1])])
        assert walks(hip, s) == [before[0] + on * (new - 1), before[1]]
        if on:
            assert np.array_equal(stepped, made["dump"])
        else:
            assert rel(made["dump"], stepped.astype(np.float64)) < tol / 2
    s.set_walks(1)


def tags_begin_anew(hip, s, t, tags):
    """Tokens by walks of that many tags each, across the last tag: the bits of the same tokens with tags from the middle."""
    s.reset()
    want = feed(s, t, [4, 1])
    for left in (tags - 1, tags, 2 * tags + 1):
        s.reset()
        walk_tags_from(hip, s, 2**32 - 1 - left)
        before = walks(hip, s)
        assert np.array_equal(feed(s, t, [4, 1]), want), left
        assert walks(hip, s) == [before[0] + len(t) - 4, before[1]]


class Opener:
    """Writes a model's folder and opens its session; close() ends them all."""

    def __init__(self, hip, tmp_path, gen):
        self.hip, self.tmp_path, self.gen, self.opened = hip, tmp_path, gen, []

    def __call__(self, cfg, w=None, dtype=F32, capacity=256):
        w = self.gen.weights(cfg) if w is None else w
        s = self.hip.models.open_session(self.gen.write_folder(self.tmp_path / f"m{len(self.opened)}", cfg, w), capacity, dtype)
        self.opened.append(s)
        return s, w

    def close(self):
        for s in self.opened:
            s.close()
