"""Dense products of several tokens, one size for every tile that the launcher picks, ragged rows and tokens among them,
through the library's own launch functions (they are C++ symbols; the structures are those of csrc/dense.h).

Reference: the f32 product of the same operands.  Bound: both sides add k f32 products, each sum within
k 2^-24 sum|a b| of the exact one."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


class RowSeg(C.Structure):
    _fields_ = [("y", C.c_void_p), ("bias", C.c_void_p), ("lower", C.c_void_p), ("mul", C.c_void_p), ("mul_tok", C.c_void_p), ("mul_ld", C.c_uint32),
                ("mul_rows", C.c_uint32), ("row0", C.c_uint32), ("n", C.c_uint32), ("ld", C.c_uint32), ("act", C.c_uint16), ("out_elem", C.c_uint16)]


class RowSegs(C.Structure):
    _fields_ = [("s", RowSeg * 12), ("start", C.c_uint32 * 12), ("n_segs", C.c_uint32), ("n_rows", C.c_uint32)]


class ColSeg(C.Structure):
    _fields_ = [("gate", C.c_void_p), ("gate_ld", C.c_uint32), ("scale", C.c_float), ("k_end", C.c_uint32)]


class ColSegs(C.Structure):
    _fields_ = [("s", ColSeg * 4), ("n_segs", C.c_uint32)]


class Dense(C.Structure):
    _fields_ = [("data", C.c_void_p), ("n_rows", C.c_uint32), ("k_pad", C.c_uint32), ("ld", C.c_uint32)]


ROWS = "_Z14rmi_dense_gemmjRK8RmiDensePKvRK10RmiRowSegsjP12ihipStream_t"
RESIDUAL = "_Z23rmi_dense_gemm_residualjRK8RmiDensePKvRK10RmiColSegsPfjjP12ihipStream_t"
K_RELU_GLU = 5


def _operand(rng, n, k, elem):
    """[n, ld] as the library wants it, and its values."""
    ld = k + (128 // elem if k * elem % 256 == 0 else 0)
    a = np.zeros((n, ld), np.float32)
    a[:, :k] = rng.standard_normal((n, k), dtype=np.float32)
    if elem == 4:
        return a, a[:, :k], ld
    bits = (a.view(np.uint32) >> 16).astype(np.uint16)
    return bits, (bits.astype(np.uint32) << 16).view(np.float32)[:, :k], ld


def _check(got, w, x, bias=None):
    k = w.shape[1]
    want = x @ w.T
    bound = 2 * k * 2.0**-24 * (np.abs(x) @ np.abs(w).T)
    assert (np.abs(got - want) <= bound).all()


@pytest.mark.parametrize("elem,rows,k,tokens", [
    (2, 12320, 1024, 2045), (2, 4096, 4096, 2041), (2, 12272, 512, 509), (2, 2048, 1024, 1000), (2, 1040, 768, 300), (2, 80, 256, 17), (2, 96, 256, 5),
    (4, 4112, 256, 1021), (4, 2064, 512, 2040), (4, 528, 256, 90)])
def test_rows(hip, elem, rows, k, tokens):
    H = hip.hip
    rng = np.random.default_rng(rows + tokens)
    w, wv, ld = _operand(rng, rows, k, elem)
    x, xv, _ = _operand(rng, tokens, k, elem)
    d_w, d_x, d_y = H.DeviceBuffer.from_array(w), H.DeviceBuffer.from_array(x), H.DeviceBuffer(rows * tokens * 4)
    segs = RowSegs()
    cut = rows // 2 // 16 * 16  # two segments, plain f32 rows
    for i, (a, b) in enumerate(((0, cut), (cut, rows))):
        segs.s[i] = RowSeg(d_y.ptr + a * 4, None, None, None, None, 0, 0, a, b - a, rows, 0, 0)
        segs.start[i] = a
    segs.start[2:] = [rows] * 10
    segs.n_segs, segs.n_rows = 2, rows
    fn = getattr(H.lib, ROWS)
    assert fn(C.c_uint32(elem), C.byref(Dense(d_w.ptr, rows, k, ld)), C.c_void_p(d_x.ptr), C.byref(segs), C.c_uint32(tokens), None) == 0
    H.check(H.lib.rmi_hip_synchronize())
    _check(d_y.to_array(np.float32, (tokens, rows)), wv, xv)


@pytest.mark.parametrize("elem,rows,k,tokens", [
    (2, 12288, 1024, 2045), (2, 4096, 4096, 2041), (2, 4100, 512, 1025), (2, 2048, 1024, 1000), (2, 1001, 512, 130), (4, 4096, 512, 1021)])
def test_residual_column_segments(hip, elem, rows, k, tokens):
    """x += gate * scale * (W a), two column segments, the first with a gate of its own and the second with one for all tokens."""
    H = hip.hip
    rng = np.random.default_rng(rows + k)
    padded = (rows + 15) // 16 * 16
    w, wv, ld = _operand(rng, padded, k, elem)
    a, av, _ = _operand(rng, tokens, k, elem)
    x = rng.standard_normal((tokens, rows), dtype=np.float32)
    gate, one = rng.uniform(0, 1, (tokens, rows)).astype(np.float32), rng.uniform(0, 1, rows).astype(np.float32)
    bufs = [H.DeviceBuffer.from_array(v) for v in (w, a, x, gate, one)]
    segs = ColSegs()
    half = k // 2 // 256 * 256
    segs.s[0], segs.s[1], segs.n_segs = ColSeg(bufs[3].ptr, rows, 0.5, half), ColSeg(bufs[4].ptr, 0, 2.0, k), 2
    fn = getattr(H.lib, RESIDUAL)
    assert fn(C.c_uint32(elem), C.byref(Dense(bufs[0].ptr, padded, k, ld)), C.c_void_p(bufs[1].ptr), C.byref(segs), C.c_void_p(bufs[2].ptr),
              C.c_uint32(rows), C.c_uint32(tokens), None) == 0
    H.check(H.lib.rmi_hip_synchronize())
    got, wv = bufs[2].to_array(np.float32, (tokens, rows)), wv[:rows]
    want = x + 0.5 * gate * (av[:, :half] @ wv[:, :half].T) + 2.0 * one * (av[:, half:] @ wv[:, half:].T)
    bound = 2 * k * 2.0**-24 * 2.0 * (np.abs(av) @ np.abs(wv).T) + 2.0**-22 * (np.abs(x) + np.abs(want))
    assert (np.abs(got - want) <= bound).all()


@pytest.mark.parametrize("elem,rows,k,tokens", [(2, 12288, 512, 1021), (2, 24576, 1024, 2045), (2, 2048, 512, 600), (4, 4096, 256, 300)])
def test_relu_pairs(hip, elem, rows, k, tokens):
    """Rows in (gate, up) pairs: relu(gate) * up, in the model's element type."""
    H = hip.hip
    rng = np.random.default_rng(rows)
    w, wv, ld = _operand(rng, rows, k, elem)
    x, xv, _ = _operand(rng, tokens, k, elem)
    d_w, d_x, d_y = H.DeviceBuffer.from_array(w), H.DeviceBuffer.from_array(x), H.DeviceBuffer(rows // 2 * tokens * elem)
    segs = RowSegs()
    segs.s[0] = RowSeg(d_y.ptr, None, None, None, None, 0, 0, 0, rows, rows // 2, K_RELU_GLU, 1)
    segs.start[1:] = [rows] * 11
    segs.n_segs, segs.n_rows = 1, rows
    fn = getattr(H.lib, ROWS)
    assert fn(C.c_uint32(elem), C.byref(Dense(d_w.ptr, rows, k, ld)), C.c_void_p(d_x.ptr), C.byref(segs), C.c_uint32(tokens), None) == 0
    H.check(H.lib.rmi_hip_synchronize())
    if elem == 2:
        got = (d_y.to_array(np.uint16, (tokens, rows // 2)).astype(np.uint32) << 16).view(np.float32)
    else:
        got = d_y.to_array(np.float32, (tokens, rows // 2))
    z, size = xv @ wv.T, np.abs(xv) @ np.abs(wv).T
    gate, up = np.maximum(z[:, 0::2], 0), z[:, 1::2]
    err = 2 * k * 2.0**-24 * size
    bound = err[:, 0::2] * np.abs(up) + err[:, 1::2] * gate + err[:, 0::2] * err[:, 1::2] + 2.0**(-8 if elem == 2 else -22) * np.abs(gate * up)
    assert (np.abs(got - gate * up) <= bound).all()
