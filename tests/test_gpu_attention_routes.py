"""Attention of several tokens, a size for every way the launcher takes (csrc/seq_mixers.hip): heads that fill a kernel's bucket
and narrower ones, few workgroups and many, keys divided over workgroups and not, keys of an earlier pass in front.  Through
the library's own launch function (a C++ symbol; the structures are those of csrc/seq_mixers.h), without convolution, rotation,
norm and gate, so that the projected rows are queries, keys and values.

Reference: softmax(scale q k) v in 64 bits.  Bound: a score is a sum of dim f32 products, a weight's error is twice the largest
error of its scores and that of an exponential and of sums over the keys (a 2^-24 a term); in bf16 weights and results are
rounded to 8 bits."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

PASS, SCRATCH = "_Z13rmi_attn_passjRK12RmiAttnShapeRK11RmiAttnArgsP12ihipStream_t", "_Z22rmi_attn_scratch_bytesRK12RmiAttnShape"


class Shape(C.Structure):
    _fields_ = [(n, C.c_uint32) for n in ("heads", "kv_heads", "dim", "vdim", "dk_pad", "dv_pad", "taps", "rot_dims")] + [
        ("scale", C.c_float), ("eps", C.c_float), ("capacity", C.c_uint32), ("window", C.c_uint32), ("v_norm", C.c_bool)]


class Args(C.Structure):
    _fields_ = [(n, C.c_void_p) for n in ("u", "hist_in", "hist_out", "conv", "cos_t", "sin_t", "q", "k_cache", "v_cache", "gate", "out")] + [
        (n, C.c_uint32) for n in ("out_ld", "pos0", "n_tokens")] + [("scratch", C.c_void_p)]


def _pad(n, to):
    return (n + to - 1) // to * to


@pytest.mark.parametrize("elem,heads,kv_heads,dim,pos0,tokens", [
    (2, 32, 8, 128, 0, 2045), (2, 16, 8, 128, 0, 1501), (2, 16, 8, 128, 0, 300), (2, 16, 8, 80, 0, 2045), (2, 16, 8, 80, 0, 300),
    (2, 16, 8, 64, 0, 2045), (2, 16, 8, 160, 0, 1201), (2, 8, 8, 160, 0, 300), (2, 16, 8, 256, 0, 701), (2, 16, 16, 160, 0, 200),
    (2, 16, 16, 160, 1000, 200), (2, 16, 16, 256, 0, 200), (2, 16, 16, 48, 1000, 200), (4, 16, 8, 80, 0, 701), (4, 16, 8, 80, 0, 200),
    (4, 16, 8, 48, 0, 701), (4, 16, 8, 160, 0, 401), (4, 16, 8, 128, 0, 401), (4, 16, 16, 160, 1000, 200), (4, 16, 16, 128, 1000, 200)])
def test_attention(hip, elem, heads, kv_heads, dim, pos0, tokens):
    H = hip.hip
    rng = np.random.default_rng(heads + dim + tokens)
    total, channels, group = pos0 + tokens, (heads + 2 * kv_heads) * dim, heads // kv_heads
    u = rng.standard_normal((total, channels), dtype=np.float32)
    if elem == 2:
        u = (u.view(np.uint32) & 0xFFFF0000).view(np.float32)
    s = Shape(heads, kv_heads, dim, dim, _pad(dim, 32), _pad(dim, 16), 1, 0, dim**-0.5, 1e-6, _pad(total, 32), 0, False)
    size = getattr(H.lib, SCRATCH)
    size.restype = C.c_size_t
    d_u, ones = H.DeviceBuffer.from_array(u), H.DeviceBuffer.from_array(np.ones(channels, np.float32))
    hist, q = H.DeviceBuffer(channels * 4), H.DeviceBuffer(heads * total * s.dk_pad * elem)
    # (caches start as zeros: a row that is not filled yet has weight zero, whatever finite value it holds)
    keys, values = (H.DeviceBuffer.from_array(np.zeros(kv_heads * s.capacity * pad * elem, np.uint8)) for pad in (s.dk_pad, s.dv_pad))
    out = H.DeviceBuffer(total * heads * dim * elem)
    scratch = H.DeviceBuffer.from_array(np.zeros(size(C.byref(s)) // 4 + 1, np.uint32))
    for first, n in ((0, pos0), (pos0, tokens)):
        if n:
            a = Args(d_u.ptr + first * channels * 4, hist.ptr, hist.ptr, ones.ptr, ones.ptr, ones.ptr, q.ptr, keys.ptr, values.ptr, None,
                     out.ptr + first * heads * dim * elem, heads * dim, first, n, scratch.ptr)
            assert getattr(H.lib, PASS)(C.c_uint32(elem), C.byref(s), C.byref(a), None) == 0
            H.check(H.lib.rmi_hip_synchronize())
    got = out.to_array(np.uint16 if elem == 2 else np.float32, (total, heads, dim))
    if elem == 2:
        got = (got.astype(np.uint32) << 16).view(np.float32)
    at = np.unique(np.r_[pos0, pos0 + 1, total - 1, rng.integers(pos0, total, 40)])
    seen = np.arange(total)[None, :] <= at[:, None]
    u = u.astype(np.float64).reshape(total, -1, dim)
    for h in range(heads):
        qh, kh, vh = u[at, h], u[:, heads + h // group], u[:, heads + kv_heads + h // group]
        z = np.where(seen, qh @ kh.T * s.scale, -np.inf)
        w = np.exp(z - z.max(1, keepdims=True))
        w /= w.sum(1, keepdims=True)
        want, size_v = w @ vh, w @ np.abs(vh)
        score = 2.0**-24 * (dim + 2) * s.scale * (np.abs(qh) @ np.abs(kh).T).max()
        bound = size_v * (2 * score + 2.0**-24 * (2 * total + 32) + (2.0**-8 if elem == 2 else 0)) + (2.0**-8 if elem == 2 else 2.0**-22) * np.abs(want)
        assert (np.abs(got[at, h] - want) <= bound).all(), (h, np.abs(got[at, h] - want).max(), bound.min())
