"""What a user of this framework has it do, as timed cases: products of quantized weights (what a host that keeps its own
loop calls) and whole decoder sessions.  `listed` names the cases, `draw` makes more of the same ranges, `prepare` / `run`
are a user's program before and during the call, `exact` is the same computation in 64 bits with torch alone.

Kinds of case:
  linear       one product on device buffers: the activation's quantizer, then the product (weights Q8_0, Q4_0, Q4_K, Q6_K)
  host         `Kernel::forward_batched` on host slices
  projections  every product of a Qwen3-0.6B token-step in one grouped launch
  qwen3        a Qwen3 Q8_0 session: greedy generation behind a prompt
  ruvenex, vogizen   model-folder sessions: a prompt, then tokens one by one that the caller chose from the logits
"""
import ctypes as C
import importlib
import os
import shutil
import tempfile

import numpy as np
import torch

rmi = importlib.import_module("rust-model-inference_amd")

# The shapes of this repository's benchmark: Qwen3-0.6B / 1.7B / 8B layers.
WIDTHS = {"0.6b": (1024, 3072, 16, 8), "1.7b": (2048, 6144, 16, 8), "8b": (4096, 12288, 32, 8)}  # width, ff, heads, kv heads
DIM, EPS, WINDOW = 128, 1e-6, 1024
RANKS = {"0.6b": (768, 256, 64), "1.7b": (1024, 512, 128), "8b": (1536, 512, 256)}  # q_rank, kv_rank, token-side inputs


def listed():
    return [
        # one token through one FFN matrix: the smallest call of a host that keeps its own decode loop
        {"name": "q8_0 token", "kind": "linear", "quant": "q8_0", "n_in": 1024, "n_out": 3072, "tokens": 1},
        # the crate's own call, host slices in and out, for a handful of sequences decoded together (odd number)
        {"name": "q8_0 host batch", "kind": "host", "n_in": 2048, "n_out": 6144, "tokens": 13},
        # the weights of a whole token-step streamed once: what decoding costs in memory traffic
        {"name": "q8_0 projections", "kind": "projections", "tokens": 1},
        # prefill of a stacked gate|up matrix
        {"name": "q8_0 prefill", "kind": "linear", "quant": "q8_0", "n_in": 1024, "n_out": 6144, "tokens": 512},
        # prefill of a K-quant down projection, a ragged number of tokens
        {"name": "q4_k prefill", "kind": "linear", "quant": "q4_k", "n_in": 6144, "n_out": 2048, "tokens": 1000},
        # the vocabulary projection of a K-quant file (its head is Q6_K)
        {"name": "q6_k head", "kind": "linear", "quant": "q6_k", "n_in": 1024, "n_out": 151936, "tokens": 1},
        # a turn of chat with Qwen3-0.6B: a prompt and an answer
        {"name": "qwen3 chat", "kind": "qwen3", "size": "0.6b", "layers": 28, "vocab": 151936, "prompt": 512, "new": 32},
        # a long document in front of the question
        {"name": "qwen3 long prompt", "kind": "qwen3", "size": "0.6b", "layers": 28, "vocab": 151936, "prompt": 1999, "new": 1},
        # a turn with a Ruvenex model of Qwen3-0.6B's size whose caller samples by itself
        {"name": "ruvenex chat", "kind": "ruvenex", "size": "0.6b", "layers": 28, "vocab": 151936, "prompt": 128, "new": 24, "dtype": "bfloat16"},
        # a prompt through layers of an 8B model: matrix products and attention
        {"name": "ruvenex prompt", "kind": "ruvenex", "size": "8b", "layers": 2, "vocab": 32768, "prompt": 2048, "new": 0, "dtype": "bfloat16"},
        # a prompt of twice the window and a few tokens: delta rule, latent attention, loop
        {"name": "vogizen prompt", "kind": "vogizen", "size": "1.7b", "layers": 4, "vocab": 32768, "prompt": 2045, "new": 4, "dtype": "bfloat16"},
        # the same model in true f32, a turn of chat
        {"name": "vogizen f32 chat", "kind": "vogizen", "size": "1.7b", "layers": 4, "vocab": 32768, "prompt": 300, "new": 16, "dtype": "float32"},
    ]


def draw(rng):
    def log(a, b):
        return min(b, int(round(a * (b / a) ** rng.random())))

    kind = rng.choice(["linear", "linear", "host", "projections", "qwen3", "qwen3", "ruvenex", "vogizen"])
    if kind == "linear":
        quant = rng.choice(["q8_0", "q8_0", "q4_k", "q6_k", "q4_0"])
        n_in = 256 * log(2, 48)
        return {"kind": kind, "quant": quant, "n_in": n_in, "n_out": min(log(500, 32000), (64 << 20) // n_in),
                "tokens": rng.choice([rng.randint(1, 8), log(9, 2048)]) if quant in ("q8_0", "q4_k") else rng.randint(1, 8)}
    if kind == "host":
        return {"kind": kind, "n_in": 32 * log(16, 256), "n_out": log(500, 12000), "tokens": log(1, 300)}
    if kind == "projections":
        return {"kind": kind, "tokens": rng.randint(2, 8)}
    if kind == "qwen3":
        size = rng.choice(["0.6b", "0.6b", "1.7b"])
        return {"kind": kind, "size": size, "layers": rng.randint(2, 28 if size == "0.6b" else 8), "vocab": rng.choice([151936, 32768]),
                "prompt": log(1, 1900), "new": log(1, 48)}
    c = {"kind": kind, "size": rng.choice(["0.6b", "1.7b"]), "layers": rng.randint(2, 8), "vocab": 32768, "prompt": log(1, 2500),
         "new": rng.randint(0, 24), "dtype": rng.choice(["bfloat16", "bfloat16", "bfloat16", "float32"])}
    return c


# ---- weights -------------------------------------------------------------------------------------------------------


def _generator(seed, part=0):
    g = torch.Generator("cuda")
    g.manual_seed(int(seed) * 64 + part)
    return g


def _normal(g, *shape):
    return torch.randn(shape, generator=g, device="cuda")


def _f16_bytes(x):
    return x.to(torch.float16).view(torch.uint8)


def _q8_0(w):
    """f32 [rows, n] -> (Q8_0 bytes, their values): scale amax / 127 in f16, quants rounded."""
    b = w.reshape(w.shape[0], -1, 32)
    d = (b.abs().amax(-1, keepdim=True) / 127).to(torch.float16)
    q = torch.where(d > 0, torch.round(b / d.float()), torch.zeros_like(b)).clamp(-127, 127)
    raw = torch.cat([_f16_bytes(d), q.to(torch.int8).view(torch.uint8)], -1)
    return raw.reshape(-1), (q * d.float()).reshape(w.shape)


def _q4_0(w):
    b = w.reshape(w.shape[0], -1, 32)
    top = torch.gather(b, -1, b.abs().argmax(-1, keepdim=True))
    d = (top / -8).to(torch.float16)
    q = torch.where(d != 0, torch.round(b / d.float()) + 8, torch.full_like(b, 8)).clamp(0, 15)
    u = q.to(torch.uint8)
    return torch.cat([_f16_bytes(d), u[..., :16] | (u[..., 16:] << 4)], -1).reshape(-1), ((q - 8) * d.float()).reshape(w.shape)


def _q4_k(w):
    b = w.reshape(w.shape[0], -1, 8, 32)
    low = (-b.amin(-1)).clamp(min=0)
    step = (b.amax(-1) + low) / 15
    d, m = ((x.amax(-1, keepdim=True) / 63).to(torch.float16) for x in (step, low))
    sc, mn = ((torch.round(x / y.float().clamp(min=1e-9))).clamp(0, 63) for x, y in ((step, d), (low, m)))
    s, o = (sc * d.float())[..., None], (mn * m.float())[..., None]
    q = torch.where(s > 0, torch.round((b + o) / s), torch.zeros_like(b)).clamp(0, 15)
    sc, mn, u = sc.to(torch.uint8), mn.to(torch.uint8), q.to(torch.uint8).reshape(*b.shape[:2], 4, 2, 32)
    packed = torch.cat([sc[..., :4] | (sc[..., 4:] >> 4 << 6), mn[..., :4] | (mn[..., 4:] >> 4 << 6), (sc[..., 4:] & 15) | (mn[..., 4:] & 15) << 4], -1)
    nibbles = (u[..., 0, :] | (u[..., 1, :] << 4)).flatten(-2)
    return torch.cat([_f16_bytes(d), _f16_bytes(m), packed, nibbles], -1).reshape(-1), (q * s - o).reshape(w.shape)


def _q6_k(w):
    b = w.reshape(w.shape[0], -1, 16, 16)
    step = b.abs().amax(-1) / 31
    d = (step.amax(-1, keepdim=True) / 127).to(torch.float16)
    sc = torch.round(step / d.float().clamp(min=1e-9)).clamp(0, 127)
    s = (sc * d.float())[..., None]
    q = torch.where(s > 0, torch.round(b / s), torch.zeros_like(b)).clamp(-32, 31)
    u = (q + 32).to(torch.uint8).reshape(*b.shape[:2], 2, 4, 32)  # halves of 128, each four runs of 32
    low = torch.stack([(u[..., 0, :] & 15) | (u[..., 2, :] & 15) << 4, (u[..., 1, :] & 15) | (u[..., 3, :] & 15) << 4], -2)
    high = (u[..., 0, :] >> 4) | (u[..., 1, :] >> 4) << 2 | (u[..., 2, :] >> 4) << 4 | (u[..., 3, :] >> 4) << 6
    raw = torch.cat([low.flatten(-3), high.flatten(-2), sc.to(torch.uint8), _f16_bytes(d)], -1)
    return raw.reshape(-1), (q * s).reshape(w.shape)


_FORMATS = {"q8_0": _q8_0, "q4_0": _q4_0, "q4_k": _q4_k, "q6_k": _q6_k}
_BLOCK_BYTES = {"q8_0": 34 / 32, "q4_0": 18 / 32, "q4_k": 144 / 256, "q6_k": 210 / 256}


def _matrix(g, rows, n):
    return _normal(g, rows, n) / n**0.5


def _upload(quant, raw, n_in, n_out):
    h = rmi.hip
    host = raw.cpu().numpy()
    handle = getattr(h.lib, "rmi_hip_upload_" + quant)(h.ptr(host, h._u8p), host.size, n_in, n_out)
    if not handle:
        raise h.RmiHipError(-1, h.last_error())
    return rmi.kernel._DeviceWeight(handle)


def _projection_shapes():
    s = rmi.synth
    return [(n_out, n_in) for _ in range(s.QWEN3_0_6B_LAYERS) for _, n_out, n_in in s.QWEN3_0_6B_LAYER] + [s.QWEN3_0_6B_LM_HEAD[1:]]


def _projection_parts(seed):
    """(bytes, values) of the matrices of one layer, in order, and of the vocabulary projection; every layer has the same."""
    g = _generator(seed)
    return [_q8_0(_matrix(g, *shape)) for shape in _projection_shapes()[:7] + _projection_shapes()[-1:]]


def _part_of(i):
    return i % 7 if i < 7 * rmi.synth.QWEN3_0_6B_LAYERS else 7


# ---- what a program has in hand before the call ----------------------------------------------------------------------


def prepare(case, seed):
    rmi.hip.init(0)
    state = globals()["_prepare_" + case["kind"]](case, seed)
    torch.cuda.synchronize()
    return state


def _linear_inputs(case, seed):
    w = _FORMATS[case["quant"]](_matrix(_generator(seed), case["n_out"], case["n_in"]))
    return w, _normal(_generator(seed, 1), case["tokens"], case["n_in"])


def _prepare_linear(case, seed):
    (raw, _), x = _linear_inputs(case, seed)
    n_in, n_out, tokens = case["n_in"], case["n_out"], case["tokens"]
    if case["quant"] in ("q8_0", "q4_0"):  # the activation, quantized: int8 and a scale a block
        act = [torch.empty(tokens, n_in, dtype=torch.int8, device="cuda"), torch.empty(tokens, n_in // 32, device="cuda")]
    else:  # Q8_K: scale, int8, sums of sixteen
        act = [torch.empty(tokens, n_in // 256, device="cuda"), torch.empty(tokens, n_in, dtype=torch.int8, device="cuda"),
               torch.empty(tokens, n_in // 16, dtype=torch.int16, device="cuda")]
    return dict(case=case, w=_upload(case["quant"], raw, n_in, n_out), x=x, act=act, y=torch.empty(tokens, n_out, device="cuda"))


def _host_inputs(case, seed):
    w = _q8_0(_matrix(_generator(seed), case["n_out"], case["n_in"]))
    return w, _normal(_generator(seed, 1), case["tokens"], case["n_in"])


def _prepare_host(case, seed):
    (raw, _), x = _host_inputs(case, seed)
    return dict(case=case, kernel=rmi.kernel.Q8Kernel(raw.cpu().numpy(), case["n_in"], case["n_out"]), x=x.cpu().numpy(),
                y=np.zeros((case["tokens"], case["n_out"]), np.float32))


class _Group:
    """A grouped launch and what it reads and writes."""

    def __init__(self, weights, q8, scales, ys, tokens):
        self.keep = weights, q8, scales, ys
        n = len(weights)
        at = [(C.c_void_p * n)(*v) for v in ([w.handle for w in weights], *([t.data_ptr() for t in v] for v in (q8, scales, ys)))]
        self.handle = rmi.hip.lib.rmi_hip_gemv_group_create(n, *at, tokens)
        if not self.handle:
            raise rmi.hip.RmiHipError(-1, rmi.hip.last_error())

    def __del__(self):
        if getattr(self, "handle", None):
            rmi.hip.lib.rmi_hip_gemv_group_destroy(self.handle)


def _projection_activation(seed, i, tokens, n_in):
    return _normal(_generator(seed, 1 + i % 8), 32, tokens, n_in)[i // 8]  # 197 problems, 32 to a generator


def _prepare_projections(case, seed):
    parts, tokens = [(r.cpu().numpy(), None) for r, _ in _projection_parts(seed)], case["tokens"]
    h, weights, q8, scales, ys = rmi.hip, [], [], [], []
    for i, (n_out, n_in) in enumerate(_projection_shapes()):
        raw = parts[_part_of(i)][0]
        weights.append(rmi.kernel._DeviceWeight(h.lib.rmi_hip_upload_q8_0(h.ptr(raw, h._u8p), raw.size, n_in, n_out)))
        q, s = _quantized(_projection_activation(seed, i, tokens, n_in))
        q8.append(q)
        scales.append(s)
        ys.append(torch.empty(tokens, n_out, device="cuda"))
    return dict(case=case, group=_Group(weights, q8, scales, ys, tokens), ys=ys)


def _quantized(x):
    """Q8_0 activation (x86-64 rounding): int8 quants, f32 scales that are f16 values."""
    b = x.reshape(x.shape[0], -1, 32)
    top = b.abs().amax(-1, keepdim=True)
    q = torch.where(top > 0, torch.round(b * (127 / top)), torch.zeros_like(b))
    return q.to(torch.int8).reshape(x.shape), (top / 127).to(torch.float16).float()[..., 0].contiguous()


def _qwen3_parts(case, seed):
    """(Q8_0 bytes, values) of one layer's matrices (every layer has the same), of the embedding and of the norms."""
    width, ff, heads, kv = WIDTHS[case["size"]]
    g = _generator(seed)
    shapes = {"attn_q": (heads * DIM, width), "attn_k": (kv * DIM, width), "attn_v": (kv * DIM, width), "attn_output": (width, heads * DIM),
              "ffn_gate": (ff, width), "ffn_up": (ff, width), "ffn_down": (width, ff)}
    layer = {n: _q8_0(_matrix(g, *s)) for n, s in shapes.items()}
    norms = {n: 1 + 0.1 * _normal(g, size) for n, size in (("attn_norm", width), ("ffn_norm", width), ("attn_q_norm", DIM), ("attn_k_norm", DIM),
                                                           ("output_norm", width))}
    return layer, norms, _q8_0(_normal(g, case["vocab"], width))


def _tokens(case, seed, n):
    return torch.randint(0, case["vocab"], (n,), generator=_generator(seed, 2), device="cuda").cpu().numpy().astype(np.uint32)


def _prepare_qwen3(case, seed):
    width, ff, heads, kv = WIDTHS[case["size"]]
    layer, norms, embed = _qwen3_parts(case, seed)
    meta = {"qwen3.embedding_length": width, "qwen3.block_count": case["layers"], "qwen3.attention.head_count": heads,
            "qwen3.attention.head_count_kv": kv, "qwen3.attention.key_length": DIM, "qwen3.attention.value_length": DIM,
            "qwen3.feed_forward_length": ff, "qwen3.vocab_size": case["vocab"], "qwen3.attention.layer_norm_rms_epsilon": EPS,
            "qwen3.rope.freq_base": 1e6}
    host = {n: raw.cpu().numpy() for n, (raw, _) in layer.items()}
    host.update({n: v.cpu().numpy() for n, v in norms.items()})
    tensors = {"token_embd.weight": embed[0].cpu().numpy(), "output_norm.weight": host.pop("output_norm")}
    tensors.update({f"blk.{i}.{n}.weight": a for i in range(case["layers"]) for n, a in host.items()})
    session = rmi.decode.Qwen3Session(meta, tensors, case["prompt"] + case["new"])
    return dict(case=case, session=session, prompt=_tokens(case, seed, case["prompt"]))


def _folder_config(case):
    width, ff, heads, kv = WIDTHS[case["size"]]
    if case["kind"] == "ruvenex":
        return rmi.folder.synthetic_ruvenex_config(case["layers"], width, ff, heads, kv, DIM, width // DIM, DIM, case["vocab"])
    q_rank, kv_rank, side = RANKS[case["size"]]
    kinds = "".join("ddda"[i % 4] for i in range(case["layers"]))
    return rmi.folder.synthetic_vogizen_config(kinds, width, ff, heads, DIM, q_rank, kv_rank, WINDOW, heads, heads // 2, DIM, side, case["vocab"],
                                               (0, min(4, case["layers"]), 2))


def _folder_weights(case, cfg, seed):
    """bf16 tensors by name for the whole model; layers of a kind have the same values, each its own copy in the file."""
    g, W, V = _generator(seed), cfg["width"], cfg["vocab"]

    def mat(rows, n):
        return _matrix(g, rows, n).bfloat16()

    def vec(n, mean, spread):
        return (mean + spread * _normal(g, n)).bfloat16()

    def conv(n):
        taps = 0.3 * _normal(g, n, 4)
        taps[:, 3] += 1
        return taps.bfloat16()

    def ruvenex(entry):
        a, r, ff = entry["mixer"]["left"], entry["mixer"]["right"], entry["mlp"]["ff"]
        nq, nk, nr = a["heads"] * a["dim"], a["kv_heads"] * a["dim"], r["heads"] * r["dim"]
        t = {"norm1": vec(W, 1, 0.1), "mix.left.g": mat(a["heads"], W), "mix.left.o": mat(W, nq), "mix.right.q": mat(nr, W), "mix.right.f": mat(nr, W),
             "mix.right.f.b": vec(nr, 2, 1), "mix.right.lower": (0.9 * torch.rand(nr, generator=g, device="cuda")).bfloat16(),
             "mix.right.v": mat(nr, W), "mix.right.norm": vec(r["vdim"], 1, 0.1), "mix.right.o": mat(W, nr), "mlp.up": mat(ff, W),
             "mlp.down": mat(W, ff), "rg1": mat(W, W), "rg1.b": vec(W, 0, 0.5), "rg2": mat(W, W), "rg2.b": vec(W, 0, 0.5)}
        for n, size in (("q", nq), ("k", nk), ("v", nk)):
            t.update({f"mix.left.{n}": mat(size, W), f"mix.left.{n}.conv": conv(size)})
        return t

    def vogizen(entry):
        m, ff, side = entry["mixer"], entry["mlp"]["ff"], cfg["token_side"]["dim"]
        nv = m["heads"] * m["vdim"]
        t = {"norm1": vec(W, 1, 0.1), "norm2": vec(W, 1, 0.1), "ls1": vec(W, 0.5, 0.1), "ls2": vec(W, 0.5, 0.1), "mlp.gate": mat(ff, W),
             "mlp.up": mat(ff, W), "mlp.down": mat(W, ff), "side.gate": mat(side, W), "side.proj": mat(W, side), "side.norm": vec(W, 0.3, 0.1),
             "mix.o": mat(W, nv)}
        if entry["type"] == "delta":
            nk = m["kv_heads"] * m["dim"]
            for n, size in (("q", nk), ("k", nk), ("v", nv)):
                t.update({f"mix.{n}": mat(size, W), f"mix.{n}.conv": conv(size)})
            t.update({"mix.b": mat(m["heads"], W), "mix.a": mat(m["heads"], W), "mix.A_log": vec(m["heads"], 0, 0.5),
                      "mix.dt_bias": vec(m["heads"], -2, 1), "mix.g": mat(nv, W), "mix.norm": vec(m["vdim"], 1, 0.1)})
        else:
            rq, rk = m["q_rank"], m["kv_rank"]
            t.update({"mix.dq": mat(rq, W), "mix.dq.norm": vec(rq, 1, 0.1), "mix.uq": mat(nv, rq), "mix.dkv": mat(rk, W),
                      "mix.dkv.norm": vec(rk, 1, 0.1), "mix.uk": mat(nv, rk), "mix.uv": mat(nv, rk)})
        return t

    kinds = {}
    for e in cfg["layers"]:
        if e["type"] not in kinds:
            kinds[e["type"]] = (ruvenex if case["kind"] == "ruvenex" else vogizen)(e)
    w = {"embed": mat(V, W), "final.norm": vec(W, 1, 0.1)}
    if case["kind"] == "ruvenex":
        w["head"] = mat(V, W)
    else:
        w.update({"loop.in": mat(W, 2 * W), "side.embed": mat(V, cfg["token_side"]["dim"]).repeat(1, len(cfg["layers"]))})
    w.update({f"l{i}.{n}": t for i, e in enumerate(cfg["layers"]) for n, t in kinds[e["type"]].items()})
    return w


def _prepare_folder(case, seed):
    cfg = _folder_config(case)
    w = _folder_weights(case, cfg, seed)
    host = {}

    def bits(t):
        if t.data_ptr() not in host:
            host[t.data_ptr()] = t.view(torch.int16).cpu().numpy().view(np.uint16)
        return host[t.data_ptr()]

    path = tempfile.mkdtemp(dir="/dev/shm" if os.path.isdir("/dev/shm") else None)
    try:
        rmi.folder._write(path, cfg, [(n, bits(t)) for n, t in w.items()])
        session = rmi.models.open_session(path, case["prompt"] + case["new"], case["dtype"])
    finally:
        shutil.rmtree(path)
    return dict(case=case, session=session, tokens=_tokens(case, seed, case["prompt"] + case["new"]))


_prepare_ruvenex = _prepare_vogizen = _prepare_folder


# ---- one pass ----------------------------------------------------------------------------------------------------------


def run(state):
    return globals()["_run_" + state["case"]["kind"]](state)


def _run_linear(s):
    lib, c, x, act, y = rmi.hip.lib, s["case"], s["x"], s["act"], s["y"]
    n_in, n_out, tokens, quant = c["n_in"], c["n_out"], c["tokens"], c["quant"]
    stream = torch.cuda.current_stream().cuda_stream
    at = [t.data_ptr() for t in act]
    if quant in ("q8_0", "q4_0"):
        rmi.hip.check(lib.rmi_hip_quantize_q8_0_dev(x.data_ptr(), *at, tokens, n_in, rmi.hip.ROUND_TIES_EVEN, stream))
        product, gemm = getattr(lib, f"rmi_hip_gemv_{quant}_dev"), lib.rmi_hip_gemm_q8_0_dev
    else:
        rmi.hip.check(lib.rmi_hip_quantize_row_q8_k_dev(x.data_ptr(), *at, tokens, n_in, stream))
        product, gemm = getattr(lib, f"rmi_hip_gemv_{quant}_q8k_dev"), lib.rmi_hip_gemm_q4_k_q8k_dev
    if tokens <= 8:
        rmi.hip.check(product(s["w"].handle, *at, y.data_ptr(), tokens, n_out, 0, n_out, stream))
    else:
        rmi.hip.check(gemm(s["w"].handle, *at, y.data_ptr(), tokens, n_out, stream))
    return y


def _run_host(s):
    c = s["case"]
    s["kernel"].forward_batched(s["x"], s["y"], c["n_in"], c["n_out"])
    return s["y"]


def _run_projections(s):
    rmi.hip.check(rmi.hip.lib.rmi_hip_gemv_group_run_dev(s["group"].handle, torch.cuda.current_stream().cuda_stream))
    ys = s["ys"]
    return {f"layer {i}": ys[7 * i:7 * i + 7] for i in (0, 13, 27)} | {"head": ys[-1]}


def _run_qwen3(s):
    n = len(s["prompt"])
    dumps = [n - 1] if s["case"]["new"] == 1 else [n - 1, n + s["case"]["new"] - 2]
    r = s["session"].generate(s["prompt"], s["case"]["new"], dumps)
    return {"logits": r["dump"][0], "last": r["dump"][-1], "tokens": r["tokens"], "argmax": r["argmax"], "top2": r["top2"]}


def _run_folder(s):
    session, tokens, n = s["session"], s["tokens"], s["case"]["prompt"]
    session.reset()
    out = [session.step(tokens[:n], want=[n - 1])]
    for t in tokens[n:]:
        out.append(session.step([t], want=[0]))
    return {"logits": np.concatenate(out)}


_run_ruvenex = _run_vogizen = _run_folder


# ---- bytes and operations that a pass cannot do without -----------------------------------------------------------------


def _folder_macs(case, cfg):
    """(weight elements read, multiply-adds a token outside attention, (heads, window) of every attention run, state elements)."""
    W = cfg["width"]
    if case["kind"] == "ruvenex":
        a, r, ff = cfg["layers"][0]["mixer"]["left"], cfg["layers"][0]["mixer"]["right"], cfg["layers"][0]["mlp"]["ff"]
        nq, nk, nr = a["heads"] * DIM, a["kv_heads"] * DIM, r["heads"] * DIM
        m = W * (nq + 2 * nk + a["heads"] + 3 * nr + 2 * W + ff + nq + nr + ff)
        n = len(cfg["layers"])
        return n * m, n * (m + 2 * nr * DIM), [(a["heads"], a["kv_heads"], None)] * n, n * nr * DIM
    loop, n, side = cfg["loop"], len(cfg["layers"]), cfg["token_side"]["dim"]
    runs = [cfg["layers"][i] for i in [*range(loop["start"]), *list(range(loop["start"], loop["stop"])) * loop["times"], *range(loop["stop"], n)]]
    weights = macs = 2 * W * W * loop["times"]
    spans, states = [], 0
    for e in runs:
        m, rest = e["mixer"], 3 * W * e["mlp"]["ff"] + 2 * W * side
        nv = m["heads"] * DIM
        if e["type"] == "delta":
            k = W * (2 * m["kv_heads"] * DIM + 3 * nv + 2 * m["heads"]) + rest
            macs, states = macs + 3 * nv * DIM, states + nv * DIM
        else:
            k = W * (m["q_rank"] + m["kv_rank"] + nv) + nv * m["q_rank"] + 2 * nv * m["kv_rank"] + rest
            spans.append((m["heads"], m["heads"], WINDOW))
        weights, macs = weights + k, macs + k
    return weights, macs, spans, states


def _seen(n, first, window):
    """Keys that positions first .. first + n - 1 read together."""
    w = window or 1 << 40
    return sum(min(p + 1, w) for p in range(first, first + n))


def work(case):
    if case["kind"] in ("linear", "host"):
        n_in, n_out, t = case["n_in"], case["n_out"], case["tokens"]
        return {"bytes": n_in * n_out * _BLOCK_BYTES[case.get("quant", "q8_0")] + 4 * t * (n_in + n_out), "flops": 2 * n_in * n_out * t}
    if case["kind"] == "projections":
        s = _projection_shapes()
        return {"bytes": sum(rmi.synth.q8_0_gemv_bytes(o, i, case["tokens"]) for o, i in s), "flops": 2 * case["tokens"] * sum(o * i for o, i in s)}
    n, new, vocab = case["prompt"], case["new"], case["vocab"]
    if case["kind"] == "qwen3":
        width, ff, heads, kv = WIDTHS[case["size"]]
        weights = case["layers"] * (width * DIM * 2 * (heads + kv) + 3 * width * ff)
        steps = n + new - 1
        flops = 2 * weights * steps + 4 * case["layers"] * heads * DIM * _seen(steps, 0, None) + 2 * width * vocab * steps  # every step's argmax
        cache = 4 * kv * DIM * case["layers"] * (n + _seen(new - 1, n, None))
        return {"bytes": new * 34 / 32 * (weights + width * vocab) + cache, "flops": flops}
    cfg = _folder_config(case)
    weights, macs, spans, states = _folder_macs(case, cfg)
    elem, W = 2 if case["dtype"] == "bfloat16" else 4, cfg["width"]
    flops = 2 * macs * (n + new) + sum(4 * h * DIM * _seen(n + new, 0, w) for h, _, w in spans) + 2 * (1 + new) * W * vocab
    cache = sum(2 * elem * kv * DIM * (n + _seen(new, n, w)) for _, kv, w in spans) + 8 * states * (1 + new)
    return {"bytes": (1 + new) * elem * (weights + W * vocab) + cache, "flops": flops}


# Products in a host's accumulation order and the Qwen3 session are the same bits from one version to the next: that is
# what this framework promises.  The Q4_K product on the matrix cores promises a tolerance (f32 sums, exact integers).
# Model folders: bf16 operands with f32 sums, or f32 throughout, through all layers.
def tolerance(case):
    if case["kind"] == "linear" and case["quant"] == "q4_k" and case["tokens"] > 8:
        return {"rel": 1e-6, "max": 1e-5}
    if case["kind"] in ("ruvenex", "vogizen"):
        return {"rel": 2e-2, "max": 0.1} if case["dtype"] == "bfloat16" else {"rel": 2e-5, "max": 2e-4}
    return "exact"


# ---- the same in 64 bits ---------------------------------------------------------------------------------------------


def exact(case, seed):
    with torch.no_grad():
        return globals()["_exact_" + case["kind"]](case, seed)


def _q8_0_values(x, k=32):
    """f64 activations rounded to Q8_0 (k = 32) or Q8_K (k = 256) and back."""
    b = x.reshape(*x.shape[:-1], -1, k)
    if k == 256:
        top = torch.gather(b, -1, b.abs().argmax(-1, keepdim=True))
        d = top / -127
        return (torch.round(torch.where(top != 0, b / d, torch.zeros_like(b))).clamp(max=127) * d).reshape(x.shape)
    d = b.abs().amax(-1, keepdim=True) / 127
    return (torch.round(torch.where(d > 0, b / d, torch.zeros_like(b))) * d.to(torch.float16).double()).reshape(x.shape)


def _exact_linear(case, seed):
    (_, w), x = _linear_inputs(case, seed)
    a = _q8_0_values(x.double(), 32 if case["quant"] in ("q8_0", "q4_0") else 256)
    return torch.cat([a @ part.double().T for part in w.split(16384)], -1)


def _exact_host(case, seed):
    (_, w), x = _host_inputs(case, seed)
    return (_q8_0_values(x.double()) @ w.double().T).cpu().numpy()


def _exact_projections(case, seed):
    parts, shapes = _projection_parts(seed), _projection_shapes()

    def product(i):
        x = _q8_0_values(_projection_activation(seed, i, case["tokens"], shapes[i][1]).double())
        return torch.cat([x @ part.double().T for part in parts[_part_of(i)][1].split(16384)], -1)

    return {f"layer {i}": [product(k) for k in range(7 * i, 7 * i + 7)] for i in (0, 13, 27)} | {"head": product(len(shapes) - 1)}


def _rms(x, weight=None, eps=EPS):
    y = x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps)
    return y if weight is None else y * weight


def _attend(q, k, v, scale, window=None):
    """q [T, H, d], k, v [T, G, d]: causal softmax attention, the last `window` positions of each; a head at a time."""
    T, H = q.shape[:2]
    p = torch.arange(T, device=q.device)
    hidden = p[None, :] > p[:, None]
    if window:
        hidden |= p[None, :] <= p[:, None] - window
    out = []
    for h in range(H):
        g = h // (H // k.shape[1])
        s = (q[:, h] @ k[:, g].T) * scale
        out.append(torch.softmax(s.masked_fill(hidden, -float("inf")), -1) @ v[:, g])
    return torch.stack(out, 1)


def _exact_qwen3(case, seed):
    """The logits behind the prompt; what follows depends on ties and has no value of its own."""
    width, ff, heads, kv = WIDTHS[case["size"]]
    layer, norms, embed = _qwen3_parts(case, seed)
    w = {n: v.double() for n, (_, v) in layer.items()}
    norms = {n: v.double() for n, v in norms.items()}
    tokens = torch.from_numpy(_tokens(case, seed, case["prompt"]).astype(np.int64)).cuda()
    x = embed[1][tokens].double()
    T = len(tokens)
    angle = torch.arange(T, device="cuda", dtype=torch.float64)[:, None] * 1e6 ** (-torch.arange(0, DIM, 2, device="cuda", dtype=torch.float64) / DIM)
    cos, sin = angle.cos()[:, None], angle.sin()[:, None]

    def rope(u):
        a, b = u.chunk(2, -1)
        return torch.cat([a * cos - b * sin, a * sin + b * cos], -1)

    def f16(u):
        return u.to(torch.float16).double()

    for _ in range(case["layers"]):
        h = _q8_0_values(_rms(x, norms["attn_norm"]))
        q, k, v = ((h @ w["attn_" + n].T).reshape(T, -1, DIM) for n in "qkv")
        q, k = f16(rope(_rms(q, norms["attn_q_norm"]))), f16(rope(_rms(k, norms["attn_k_norm"])))
        a = _attend(q, k, f16(v), DIM**-0.5)
        x = x + _q8_0_values(a.reshape(T, -1)) @ w["attn_output"].T
        h = _q8_0_values(_rms(x, norms["ffn_norm"]))
        g = h @ w["ffn_gate"].T
        x = x + _q8_0_values(g * torch.sigmoid(g) * (h @ w["ffn_up"].T)) @ w["ffn_down"].T
    h = _q8_0_values(_rms(x[-1:], norms["output_norm"]))
    logits = torch.cat([h @ part.double().T for part in embed[1].split(16384)], -1)[0]
    return {"logits": logits.cpu().numpy(), "last": None, "tokens": None, "argmax": None, "top2": None}


def _conv(u, taps):
    n = taps.shape[1]
    padded = torch.cat([u.new_zeros(n - 1, u.shape[1]), u])
    return sum(taps[:, j] * padded[j:j + u.shape[0]] for j in range(n))


def _silu(z):
    return z * torch.sigmoid(z)


def _gelu(z):
    return torch.nn.functional.gelu(z, approximate="tanh")


def _ruvenex_layer(x, w, p, c):
    T, h = x.shape[0], _rms(x, w(p + "norm1"))
    a, r, m = c["mixer"]["left"], c["mixer"]["right"], p + "mix."
    q, k, v = (_conv(h @ w(m + "left." + n).T, w(m + f"left.{n}.conv")).reshape(T, -1, DIM) for n in "qkv")
    turned, i = a["rot"]["dims"], torch.arange(0, a["rot"]["dims"], 2, device="cuda", dtype=torch.float64)
    angle = torch.arange(T, device="cuda", dtype=torch.float64)[:, None] * a["rot"]["base"] ** (-i / turned)
    cos, sin = angle.cos()[:, None], angle.sin()[:, None]

    def rope(u):
        e, o = u[..., 0:turned:2], u[..., 1:turned:2]
        return torch.cat([torch.stack([e * cos - o * sin, o * cos + e * sin], -1).flatten(-2), u[..., turned:]], -1)

    left = _attend(rope(q), rope(k), _rms(v), a["scale"]) * torch.sigmoid(h @ w(m + "left.g").T)[..., None]
    left = left.reshape(T, -1) @ w(m + "left.o").T
    q = _silu(h @ w(m + "right.q").T).reshape(T, -1, DIM)
    low = w(m + "right.lower")
    f = (low + (1 - low) * torch.sigmoid(h @ w(m + "right.f").T + w(m + "right.f.b"))).reshape(T, -1, DIM)
    v = (h @ w(m + "right.v").T).reshape(T, -1, DIM)
    S, out = x.new_zeros(r["heads"], DIM, DIM), []
    for t in range(T):
        S = f[t][:, :, None] * S + (1 - f[t])[:, :, None] * v[t][:, None, :]
        out.append((q[t][:, None, :] @ S)[:, 0])
    right = _rms(torch.stack(out), w(m + "right.norm")).reshape(T, -1) @ w(m + "right.o").T
    mixed = c["mixer"]["left_scale"] * left + c["mixer"]["right_scale"] * right
    x = x + torch.sigmoid(h @ w(p + "rg1").T + w(p + "rg1.b")) * mixed
    return x + torch.sigmoid(h @ w(p + "rg2").T + w(p + "rg2.b")) * (_gelu(h @ w(p + "mlp.up").T) @ w(p + "mlp.down").T)


def _layer_norm(x, weight):
    return torch.nn.functional.layer_norm(x, x.shape[-1:], eps=EPS) * weight


def _delta(h, w, p, c):
    T, H, G = h.shape[0], c["heads"], c["kv_heads"]
    q, k, v = (_silu(_conv(h @ w(p + n).T, w(p + n + ".conv"))).reshape(T, -1, DIM) for n in "qkv")
    q, k = (u * torch.rsqrt((u * u).sum(-1, keepdim=True) + 1e-6) for u in (q, k))
    share = torch.arange(H, device="cuda") // (H // G)
    q, k = q[:, share] * DIM**-0.5, k[:, share]
    beta = torch.sigmoid(h @ w(p + "b").T)
    g = torch.exp(-torch.exp(w(p + "A_log")) * torch.nn.functional.softplus(h @ w(p + "a").T + w(p + "dt_bias"), threshold=1e9))
    S, out = h.new_zeros(H, DIM, DIM), []
    for t in range(T):
        S = g[t][:, None, None] * S
        u = beta[t][:, None] * (v[t] - (k[t][:, None, :] @ S)[:, 0])
        S = S + k[t][:, :, None] * u[:, None, :]
        out.append((q[t][:, None, :] @ S)[:, 0])
    o = _rms(torch.stack(out), w(p + "norm")).reshape(T, -1) * _silu(h @ w(p + "g").T)
    return o @ w(p + "o").T


def _latent(h, w, p, c):
    T = h.shape[0]
    q = _rms(h @ w(p + "dq").T, w(p + "dq.norm")) @ w(p + "uq").T
    lat = _rms(h @ w(p + "dkv").T, w(p + "dkv.norm"))
    q, k, v = (u.reshape(T, -1, DIM) for u in (q, lat @ w(p + "uk").T, lat @ w(p + "uv").T))
    return _attend(q, k, v, c["scale"], c["mask"]["size"]).reshape(T, -1) @ w(p + "o").T


def _vogizen_layers(x, w, cfg, tokens):
    T, W, n, loop = len(tokens), cfg["width"], len(cfg["layers"]), cfg["loop"]
    i = torch.arange(W, device="cuda")
    a = torch.arange(T, device="cuda", dtype=torch.float64)[:, None] * 10000.0 ** (-2.0 * (i // 2) / W)
    x = x0 = x + torch.where(i % 2 == 0, a.sin(), a.cos())
    side = cfg["token_side"]["dim"]
    inner = list(range(loop["start"], loop["stop"]))
    runs = [(i, False) for i in range(loop["start"])] + [(i, i == loop["start"]) for _ in range(loop["times"]) for i in inner]
    for i, begins in runs + [(i, False) for i in range(loop["stop"], n)]:
        c, p = cfg["layers"][i], f"l{i}."
        if begins:
            x = torch.cat([x, x0], 1) @ w("loop.in").T
        mixer = _delta if c["type"] == "delta" else _latent
        x = x + w(p + "ls1") * mixer(_layer_norm(x, w(p + "norm1")), w, p + "mix.", c["mixer"])
        h = _layer_norm(x, w(p + "norm2"))
        x = x + w(p + "ls2") * ((torch.relu(h @ w(p + "mlp.gate").T) * (h @ w(p + "mlp.up").T)) @ w(p + "mlp.down").T)
        e = w("side.embed", tokens)[:, i * side:(i + 1) * side]
        x = x + _rms((_gelu(x @ w(p + "side.gate").T) * e) @ w(p + "side.proj").T, w(p + "side.norm"))
    return x


def _exact_folder(case, seed):
    cfg = _folder_config(case)
    weights = _folder_weights(case, cfg, seed)

    def w(name, rows=None):
        return (weights[name] if rows is None else weights[name][rows]).double()

    tokens = torch.from_numpy(_tokens(case, seed, case["prompt"] + case["new"]).astype(np.int64)).cuda()
    x = w("embed", tokens)
    if case["kind"] == "ruvenex":
        for i, c in enumerate(cfg["layers"]):
            x = _ruvenex_layer(x, w, f"l{i}.", c)
        head, h = "head", _rms(x[case["prompt"] - 1:], w("final.norm"))
    else:
        x = _vogizen_layers(x, w, cfg, tokens)
        head, h = "embed", _layer_norm(x[case["prompt"] - 1:], w("final.norm"))
    return {"logits": torch.cat([h @ part.double().T for part in weights[head].split(16384)], -1).cpu().numpy()}


_exact_ruvenex = _exact_vogizen = _exact_folder
