"""Prompt passes of the Qwen3 session over the range of contexts: in larger passes 32 positions of a head share a
workgroup of the attention, so lengths on both sides of a tile, of a 128-key turn and of a pass, with the keys of earlier passes in
front.  Every position its own step is the reference (held to the CPU loop by test_gpu_decode_device.py): all bits equal."""
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads,kv_heads,n_prompt,per_pass", [
    (8, 4, 2, True), (8, 4, 16, True), (8, 4, 17, True), (3, 3, 65, True), (8, 2, 127, 33), (4, 1, 512, True), (4, 4, 513, True),
    (2, 1, 700, 129), (4, 2, 1300, True), (2, 2, 2100, True),
    # up to 1024 positions times heads (256 compute units) a workgroup takes one position, beyond that 32
    (8, 4, 128, True), (8, 4, 129, True), (64, 8, 16, True), (64, 8, 17, True), (64, 16, 33, True), (32, 8, 700, 40), (64, 8, 300, 63), (32, 4, 700, 30)])
def test_passes_have_the_bits_of_single_steps(hip, tmp_path, heads, kv_heads, n_prompt, per_pass):
    path = os.path.join(str(tmp_path), "m.gguf")
    hip.gguf.write_synthetic_qwen3(path, seed=heads, n_layer=2, n_embd=256, n_head=heads, n_head_kv=kv_heads, head_dim=128, n_ff=512, vocab=1000,
                                   n_ctx=4096)
    f = hip.gguf.GGUFFile(path)
    session = hip.decode.Qwen3Session(f.metadata, {name: t[2] for name, t in f.tensors.items()}, capacity=n_prompt + 4)
    prompt = np.random.default_rng(n_prompt).integers(0, 1000, n_prompt, dtype=np.uint32)
    dumps = sorted({0, n_prompt // 2, n_prompt - 1, n_prompt, n_prompt + 2})
    session.set_prompt_passes(per_pass)
    fast = session.generate(prompt, 4, dump_steps=dumps)
    session.set_prompt_passes(False)
    slow = session.generate(prompt, 4, dump_steps=dumps)
    session.close()
    assert np.array_equal(fast["tokens"], slow["tokens"]) and np.array_equal(fast["argmax"], slow["argmax"])
    assert np.array_equal(fast["top2"].view(np.uint32), slow["top2"].view(np.uint32))
    assert np.array_equal(fast["dump"].view(np.uint32), slow["dump"].view(np.uint32))


@pytest.mark.parametrize("n_prompt", [200, 300])
def test_logits_of_every_position_of_a_pass(hip, tmp_path, n_prompt):
    """A pass makes logits 128 positions at a time and hands on those asked for, here all of them."""
    path = os.path.join(str(tmp_path), "m.gguf")
    hip.gguf.write_synthetic_qwen3(path, seed=9, n_layer=2, n_embd=256, n_head=4, n_head_kv=2, head_dim=128, n_ff=512, vocab=1000, n_ctx=4096)
    f = hip.gguf.GGUFFile(path)
    session = hip.decode.Qwen3Session(f.metadata, {name: t[2] for name, t in f.tensors.items()}, capacity=n_prompt + 2)
    prompt = np.random.default_rng(4).integers(0, 1000, n_prompt, dtype=np.uint32)
    fast = session.generate(prompt, 2, dump_steps=range(n_prompt + 1))
    session.set_prompt_passes(False)
    slow = session.generate(prompt, 2, dump_steps=range(n_prompt + 1))
    session.close()
    assert np.array_equal(fast["dump"].view(np.uint32), slow["dump"].view(np.uint32))


@pytest.mark.parametrize("heads,kv_heads,n_prompt,per_pass", [
    # below and from a million products of a query and a key on (there in limbs)
    (64, 8, 95, True), (32, 8, 130, True), (64, 8, 181, True), (64, 8, 224, True), (64, 8, 225, True), (32, 8, 257, True), (8, 2, 600, True), (64, 8, 330, 161)])
@pytest.mark.parametrize("q,k,v", [(10.0, 10.0, 1.0), (40.0, 1.0, 1.0), (1.0, 1.0, 150.0), (10.0, 5.0, 400.0), (1e-5, 0.3, 1e-6)])
def test_values_at_the_edge_of_what_limbs_hold(hip, tmp_path, heads, kv_heads, n_prompt, per_pass, q, k, v):
    """Queries, keys and values times q, k, v: large scores make weights of one and of a half (a fourth limb), small factors
    subnormal f16 values; values from 127 on put their head in f64, norms from 11.2 on (40) the whole layer.  The bits are the
    same in every form; test_gpu_attn_prompt.py says which pass takes which, and has queries and keys at the edge."""
    path = os.path.join(str(tmp_path), "m.gguf")
    hip.gguf.write_synthetic_qwen3(path, seed=heads, n_layer=2, n_embd=256, n_head=heads, n_head_kv=kv_heads, head_dim=128, n_ff=256, vocab=500, n_ctx=4096)
    f = hip.gguf.GGUFFile(path)
    t = {name: np.array(x[2]) for name, x in f.tensors.items()}
    for layer in range(2):
        t[f"blk.{layer}.attn_q_norm.weight"] = t[f"blk.{layer}.attn_q_norm.weight"] * np.float32(q)
        t[f"blk.{layer}.attn_k_norm.weight"] = t[f"blk.{layer}.attn_k_norm.weight"] * np.float32(k)
        blocks = t[f"blk.{layer}.attn_v.weight"].reshape(-1, 34)
        blocks[:, :2] = (blocks[:, :2].copy().view(np.float16) * np.float16(v)).view(np.uint8)
    session = hip.decode.Qwen3Session(f.metadata, t, capacity=n_prompt + 4)
    prompt = np.random.default_rng(n_prompt).integers(0, 500, n_prompt, dtype=np.uint32)
    session.set_prompt_passes(per_pass)
    fast = session.generate(prompt, 2, dump_steps=range(n_prompt + 1))
    session.set_prompt_passes(False)
    slow = session.generate(prompt, 2, dump_steps=range(n_prompt + 1))
    session.close()
    assert np.array_equal(fast["dump"].view(np.uint32), slow["dump"].view(np.uint32))


def _put(raw, n_in, row, block, scale, quants):
    """One block of 32 of a row of Q8_0 bytes."""
    b = raw.reshape(-1, n_in // 32, 34)[row, block]
    b[:2] = np.frombuffer(np.float16(scale).tobytes(), np.uint8)
    b[2:] = np.asarray(quants, np.int8).view(np.uint8)


@pytest.mark.parametrize("seen", [True, False])
@pytest.mark.parametrize("heads,n_prompt,at", [(2, 5, 4), (2, 40, 20), (64, 17, 16), (64, 18, 2), (64, 33, 32), (64, 40, 20), (64, 40, 35), (64, 100, 80), (64, 130, 129), (64, 230, 20), (64, 230, 200), (64, 230, 229)])
def test_a_value_that_is_not_finite_counts_from_its_position_on(hip, tmp_path, heads, n_prompt, at, seen):
    """One prompt token's values overflow f16.  seen: its weight is not zero, so that its position and those behind it have
    logits that are not finite, and their number is in the error.  Otherwise every weight of it rounds to zero: 0 x inf is
    NaN, which the quantizer drops, from that position on and not before."""
    width, special = 256, 999
    path = os.path.join(str(tmp_path), "m.gguf")
    hip.gguf.write_synthetic_qwen3(path, seed=5, n_layer=1, n_embd=width, n_head=heads, n_head_kv=heads, head_dim=128, n_ff=256, vocab=1000, n_ctx=4096)
    f = hip.gguf.GGUFFile(path)
    t = {name: np.array(v[2]) for name, v in f.tensors.items()}
    # elements 0 and 1 of the stream: the special token's mark, and one that all tokens have
    for row in range(1000):
        q = t["token_embd.weight"].reshape(-1, width // 32, 34)[row, 0, 2:].view(np.int8)
        q[0], q[1] = 0, 127
    _put(t["token_embd.weight"], width, special, 0, 1.0, [127, 127] + [0] * 30)
    for row in range(0, heads * 128, 5):  # some values of every block (of nothing but NaN the largest is NaN): 500 x 127 times the mark
        _put(t["blk.0.attn_v.weight"], width, row, 0, 500.0, [127] + [0] * 31)
    if not seen:  # one element a head, of one sign in every query, of the other sign in the special token's key: scores of +-100
        for name in ("attn_q", "attn_k"):
            w = t[f"blk.0.{name}.weight"].reshape(-1, width // 32, 34)
            w[:, :, 2:] = 0
            for head in range(heads):
                _put(t[f"blk.0.{name}.weight"], width, head * 128 + 63, 0, 0.1, [-127 if name == "attn_k" else 0, 64] + [0] * 30)
            t[f"blk.0.{name}_norm.weight"] = np.full(128, 3.0, np.float32)
    session = hip.decode.Qwen3Session(f.metadata, t, capacity=n_prompt + 4)
    prompt = np.random.default_rng(n_prompt).integers(0, 999, n_prompt, dtype=np.uint32)
    prompt[at] = special

    def outcome(passes):
        session.set_prompt_passes(passes)
        try:
            r = session.generate(prompt, 1, dump_steps=range(n_prompt))
        except hip.hip.RmiHipError as e:
            return str(e)
        return r["dump"].view(np.uint32), r["argmax"], r["tokens"]

    fast, slow = outcome(True), outcome(False)
    session.close()
    if seen:
        assert f"{n_prompt - at} steps" in slow and fast == slow
    else:
        assert not isinstance(slow, str), slow
        assert all(np.array_equal(a, b) for a, b in zip(fast, slow))


def test_a_pass_whose_scores_exceed_the_scratch(hip, tmp_path):
    """64 heads' scores of 1024 positions at a capacity of 2000 are more than the 256 MB of scratch: several launches a pass."""
    heads, n_prompt = 64, 1990
    path = os.path.join(str(tmp_path), "m.gguf")
    hip.gguf.write_synthetic_qwen3(path, seed=2, n_layer=1, n_embd=64, n_head=heads, n_head_kv=8, head_dim=128, n_ff=64, vocab=500, n_ctx=4096)
    f = hip.gguf.GGUFFile(path)
    session = hip.decode.Qwen3Session(f.metadata, {name: t[2] for name, t in f.tensors.items()}, capacity=2000)
    prompt = np.random.default_rng(3).integers(0, 500, n_prompt, dtype=np.uint32)
    dumps = [0, 255, 500, 511, 512, 800, 1023, 1024, 1500, 1700, 1989, 1992]
    fast = session.generate(prompt, 4, dump_steps=dumps)
    session.set_prompt_passes(False)
    slow = session.generate(prompt, 4, dump_steps=dumps)
    session.close()
    assert np.array_equal(fast["tokens"], slow["tokens"]) and np.array_equal(fast["argmax"], slow["argmax"])
    assert np.array_equal(fast["top2"].view(np.uint32), slow["top2"].view(np.uint32))
    assert np.array_equal(fast["dump"].view(np.uint32), slow["dump"].view(np.uint32))
