"""Prompt passes of the Qwen3 session over the range of contexts: sixteen positions of a head share a workgroup of the
pass's attention, so lengths on both sides of a tile, of a 64-key turn and of a pass, with the keys of earlier passes in
front.  Every position its own step is the reference (held to the CPU loop by test_gpu_decode_device.py): all bits equal."""
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads,kv_heads,n_prompt,per_pass", [
    (8, 4, 2, True), (8, 4, 16, True), (8, 4, 17, True), (3, 3, 65, True), (8, 2, 127, 33), (4, 1, 512, True), (4, 4, 513, True),
    (2, 1, 700, 129), (4, 2, 1300, True), (2, 2, 2100, True)])
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


def test_a_pass_that_is_asked_for_more_logits_than_it_holds(hip, tmp_path):
    """64 positions' logits of a pass can be asked for; with more the pass ends early and the next one goes on."""
    path = os.path.join(str(tmp_path), "m.gguf")
    hip.gguf.write_synthetic_qwen3(path, seed=9, n_layer=2, n_embd=256, n_head=4, n_head_kv=2, head_dim=128, n_ff=512, vocab=1000, n_ctx=4096)
    f = hip.gguf.GGUFFile(path)
    session = hip.decode.Qwen3Session(f.metadata, {name: t[2] for name, t in f.tensors.items()}, capacity=202)
    prompt = np.random.default_rng(4).integers(0, 1000, 200, dtype=np.uint32)
    fast = session.generate(prompt, 2, dump_steps=range(201))
    session.set_prompt_passes(False)
    slow = session.generate(prompt, 2, dump_steps=range(201))
    session.close()
    assert np.array_equal(fast["dump"].view(np.uint32), slow["dump"].view(np.uint32))
