"""Products of several tokens whose k is divided over workgroups (csrc/dense.hip), through the library's own launch functions.
Each case asserts that it is divided, and is launched three times on the same counters: the same bits, and counters at zero behind it.

Reference and bound as in test_gpu_dense_tiles: k f32 products a side, in whatever order."""
import ctypes as C

import numpy as np
import pytest

from test_gpu_dense_tiles import PARTS, RESIDUAL, ROWS, ColSeg, ColSegs, Dense, RowSeg, RowSegs, Work, _check, _operand

pytestmark = pytest.mark.gpu

COUNTERS, SUMS = 4096, 4096 * 1024


def _work(H):
    bufs = H.DeviceBuffer.from_array(np.zeros(COUNTERS, np.uint32)), H.DeviceBuffer(SUMS * 4)
    return bufs, Work(bufs[0].ptr, bufs[1].ptr)


def _is_divided(H, elem, epilogue, rows, k, tokens):
    fn = getattr(H.lib, PARTS)
    fn.restype = C.c_uint32
    return fn(C.c_uint32(elem), C.c_int(epilogue), C.c_uint32(rows), C.c_uint32(k), C.c_uint32(tokens)) >> 16 > 1


# tiles of 16, 32 and 64 tokens; k of rounds that the parts do not share evenly; one row of tiles and more than compute units; ragged ends
@pytest.mark.parametrize("elem,rows,k,tokens", [
    (2, 1024, 6144, 128), (2, 1002, 4096, 45), (2, 64, 3328, 5), (2, 2046, 6144, 16), (2, 80, 2816, 17), (2, 4096, 12288, 61), (2, 1024, 6144, 300),
    (4, 2048, 6144, 300), (4, 1030, 1408 // 256 * 256, 33), (4, 66, 1280, 2), (4, 1000, 3072, 9), (4, 2048, 2048, 289)])
def test_residual_in_parts(hip, elem, rows, k, tokens):
    """Three column segments whose ends lie inside parts, with a gate of its own, one for all tokens, and none."""
    H = hip.hip
    assert _is_divided(H, elem, -1, rows, k, tokens)
    rng = np.random.default_rng(rows + k)
    padded = (rows + 15) // 16 * 16
    w, wv, ld = _operand(rng, padded, k, elem)
    a, av, _ = _operand(rng, tokens, k, elem)
    x = rng.standard_normal((tokens, rows), dtype=np.float32)
    gate, one = rng.uniform(0, 1, (tokens, rows)).astype(np.float32), rng.uniform(0, 1, rows).astype(np.float32)
    bufs = [H.DeviceBuffer.from_array(v) for v in (w, a, gate, one)]
    ends = k // 4 // 256 * 256 or 256, k // 4 // 256 * 256 + 256, k
    segs = ColSegs()
    segs.s[0], segs.s[1], segs.s[2] = ColSeg(bufs[2].ptr, rows, 0.5, ends[0]), ColSeg(bufs[3].ptr, 0, 2.0, ends[1]), ColSeg(None, rows, 1.0, k)
    segs.n_segs = 3
    keep, work = _work(H)
    seen = []
    for _ in range(3):
        d_x = H.DeviceBuffer.from_array(x)
        assert getattr(H.lib, RESIDUAL)(C.c_uint32(elem), C.byref(Dense(bufs[0].ptr, padded, k, ld)), C.c_void_p(bufs[1].ptr), C.byref(segs),
                                        C.c_void_p(d_x.ptr), C.c_uint32(rows), C.c_uint32(tokens), C.byref(work), None) == 0
        H.check(H.lib.rmi_hip_synchronize())
        seen.append(d_x.to_array(np.float32, (tokens, rows)))
        assert not keep[0].to_array(np.uint32, (COUNTERS,)).any()
    want, size, first = x.astype(np.float64), np.zeros((tokens, rows)), 0
    for end, g, scale in zip(ends, (gate, one, 1.0), (0.5, 2.0, 1.0)):
        want = want + scale * g * (av[:, first:end] @ wv[:rows, first:end].T)
        size = size + scale * (np.abs(av[:, first:end]) @ np.abs(wv[:rows, first:end]).T)
        first = end
    assert (np.abs(seen[0] - want) <= 2 * k * 2.0**-24 * size + 2.0**-21 * (np.abs(x) + np.abs(want))).all()
    assert all(np.array_equal(s.view(np.uint32), seen[0].view(np.uint32)) for s in seen[1:])


@pytest.mark.parametrize("elem,rows,k,tokens", [(2, 128, 4096, 300), (2, 80, 3072, 3), (4, 128, 2048, 300), (4, 112, 1280, 1000), (4, 48, 1024, 12)])
def test_rows_in_parts(hip, elem, rows, k, tokens):
    H = hip.hip
    assert _is_divided(H, elem, 0, rows, k, tokens)
    rng = np.random.default_rng(rows + tokens)
    w, wv, ld = _operand(rng, rows, k, elem)
    x, xv, _ = _operand(rng, tokens, k, elem)
    d_w, d_x = H.DeviceBuffer.from_array(w), H.DeviceBuffer.from_array(x)
    keep, work = _work(H)
    seen = []
    for _ in range(3):
        d_y = H.DeviceBuffer.from_array(np.full((tokens, rows), np.nan, np.float32))
        segs = RowSegs()
        cut = rows // 2 // 16 * 16
        for i, (a, b) in enumerate(((0, cut), (cut, rows))):
            segs.s[i] = RowSeg(d_y.ptr + a * 4, None, None, None, None, 0, 0, a, b - a, rows, 0, 0)
            segs.start[i] = a
        segs.start[2:] = [rows] * 10
        segs.n_segs, segs.n_rows = 2, rows
        assert getattr(H.lib, ROWS)(C.c_uint32(elem), C.byref(Dense(d_w.ptr, rows, k, ld)), C.c_void_p(d_x.ptr), C.byref(segs), C.c_uint32(tokens),
                                    C.byref(work), None) == 0
        H.check(H.lib.rmi_hip_synchronize())
        seen.append(d_y.to_array(np.float32, (tokens, rows)))
        assert not keep[0].to_array(np.uint32, (COUNTERS,)).any()
    _check(seen[0], wv, xv)
    assert all(np.array_equal(s.view(np.uint32), seen[0].view(np.uint32)) for s in seen[1:])
