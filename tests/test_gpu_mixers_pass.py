"""Attention and the gated recurrence of several tokens side by side (rmi_mixers_pass, csrc/seq_mixers.hip): keys divided over workgroups and
not, scans of one segment and of several, chunks with tokens missing, a pass in front.  Through the library's own launch functions.

Attention: the bits of rmi_attn_pass.  Recurrence: the sequential statement in 64 bits; an o is a sum over channels and over the tokens before
it whose factors are products of up to n gates, so its error is within (dim + 2 n) 2^-24 of the same sum of absolute values, and the norm's
root mean square is off by no more than the largest of those; bf16 results are rounded to 8 bits."""
import ctypes as C

import numpy as np
import pytest

from test_gpu_attention_routes import PASS, SCRATCH, Args, Shape

pytestmark = pytest.mark.gpu

BOTH = "_Z15rmi_mixers_passjRK12RmiAttnShapeRK11RmiAttnArgsRK13RmiRecurShapeRK12RmiRecurArgsP12ihipStream_t"
RECUR_SCRATCH = "_Z24rmi_recur_scratch_floatsRK13RmiRecurShapej"
DIM = 128


class RecurShape(C.Structure):
    _fields_ = [(n, C.c_uint32) for n in ("heads", "dim", "vdim", "d_pad", "v_pad")] + [("eps", C.c_float)]


class RecurArgs(C.Structure):
    _fields_ = [(n, C.c_void_p) for n in ("q", "f", "v", "state_in", "state_out", "norm", "out")] + [(n, C.c_uint32) for n in ("out_ld", "pos0", "n_tokens")] + [
        ("scratch", C.c_void_p)]


def _values(buf, elem, shape):
    a = buf.to_array(np.uint16 if elem == 2 else np.float32, shape)
    return (a.astype(np.uint32) << 16).view(np.float32) if elem == 2 else a


@pytest.mark.parametrize("elem,dim,vdim,passes", [
    (2, 128, 128, (2, 15)), (2, 128, 128, (128,)), (2, 126, 128, (129, 40)), (2, 127, 100, (300,)), (2, 128, 128, (1030, 5)),
    (4, 128, 128, (33, 2)), (4, 126, 128, (257,)), (4, 113, 120, (64, 300))])
def test_both_mixers(hip, elem, dim, vdim, passes):
    H = hip.hip
    rng = np.random.default_rng(dim + sum(passes))
    heads, kv_heads, r_heads, total = 4, 2, 2, sum(passes)
    channels = (heads + 2 * kv_heads) * DIM
    s = Shape(heads, kv_heads, DIM, DIM, DIM, DIM, 1, 0, DIM**-0.5, 1e-6, (total + 31) // 32 * 32, 0, True)
    rs = RecurShape(r_heads, dim, vdim, DIM, (vdim + 15) // 16 * 16, 1e-6)
    u = rng.standard_normal((total, channels), dtype=np.float32)
    q, v = rng.standard_normal((total, r_heads, dim), dtype=np.float32), rng.standard_normal((total, r_heads, vdim), dtype=np.float32)
    f = (1 - 0.3 * rng.random((total, r_heads, dim)) ** 3).astype(np.float32)
    f[rng.random(f.shape) < 0.01] = 0  # channels that forget at once
    norm = (1 + 0.1 * rng.standard_normal(vdim)).astype(np.float32)
    size, r_size = getattr(H.lib, SCRATCH), getattr(H.lib, RECUR_SCRATCH)
    size.restype = r_size.restype = C.c_size_t
    d_u, d_q, d_f, d_v, d_norm, ones = [H.DeviceBuffer.from_array(a) for a in (u, q, f, v, norm, np.ones(channels, np.float32))]
    hist, qbuf = H.DeviceBuffer(channels * 4), H.DeviceBuffer(heads * total * DIM * elem)
    width = heads * DIM + r_heads * vdim
    scratch = H.DeviceBuffer.from_array(np.zeros(size(C.byref(s)) // 4 + 1, np.uint32))
    r_scratch = H.DeviceBuffer(r_size(C.byref(rs), C.c_uint32(max(passes))) * 4)
    states = [H.DeviceBuffer.from_array(np.zeros((r_heads, DIM, rs.v_pad), np.float32)) for _ in range(2)]
    outs = []
    for both in (True, False):
        keys, values = (H.DeviceBuffer.from_array(np.zeros(kv_heads * s.capacity * DIM * elem, np.uint8)) for _ in range(2))
        out, first = H.DeviceBuffer(total * width * elem), 0
        for i, n in enumerate(passes):
            a = Args(d_u.ptr + first * channels * 4, hist.ptr, hist.ptr, ones.ptr, ones.ptr, ones.ptr, qbuf.ptr, keys.ptr, values.ptr, None,
                     out.ptr + first * width * elem, width, first, n, scratch.ptr)
            r = RecurArgs(d_q.ptr + first * r_heads * dim * 4, d_f.ptr + first * r_heads * dim * 4, d_v.ptr + first * r_heads * vdim * 4, states[i % 2].ptr,
                          states[1 - i % 2].ptr, d_norm.ptr, out.ptr + (first * width + heads * DIM) * elem, width, first, n, r_scratch.ptr)
            if both:
                assert getattr(H.lib, BOTH)(C.c_uint32(elem), C.byref(s), C.byref(a), C.byref(rs), C.byref(r), None) == 0
            else:
                assert getattr(H.lib, PASS)(C.c_uint32(elem), C.byref(s), C.byref(a), None) == 0
            H.check(H.lib.rmi_hip_synchronize())
            first += n
        outs.append(_values(out, elem, (total, width)))
        if both:
            state = states[len(passes) % 2].to_array(np.float32, (r_heads, DIM, rs.v_pad))
    assert np.array_equal(outs[0][:, :heads * DIM], outs[1][:, :heads * DIM])
    got = outs[0][:, heads * DIM:].reshape(total, r_heads, vdim)
    S, A = np.zeros((r_heads, dim, vdim)), np.zeros((r_heads, dim, vdim))
    q, f, v = (t.astype(np.float64) for t in (q, f, v))
    unit = 2.0**-24 * (dim + 2 * total)
    for t in range(total):
        k = 1 - f[t]
        S, A = f[t][:, :, None] * S + k[:, :, None] * v[t][:, None, :], f[t][:, :, None] * A + k[:, :, None] * np.abs(v[t])[:, None, :]
        o, err = np.einsum("hd,hdv->hv", q[t], S), unit * np.einsum("hd,hdv->hv", np.abs(q[t]), A)
        rms = np.sqrt((o * o).mean(-1, keepdims=True) + 1e-6)
        want = o / rms * norm
        bound = (err + np.abs(o) * (err.max(-1, keepdims=True) / rms + 2.0**-20)) / rms * np.abs(norm) + (2.0**-8 * np.abs(want) if elem == 2 else 0)
        assert (np.abs(got[t] - want) <= bound).all(), t
    assert (np.abs(state[:, :dim, :vdim] - S) <= unit * A + 1e-30).all()
