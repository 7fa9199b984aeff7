"""Products of several tokens in the x86-64 order (matmul_q8_0_vs_q8_0_avx2, src/ops/kernel/q8_0/avx2.rs:71-173): the GEMV's
token groups, of eight and of four, whole, ragged (the last group begins earlier) and with a launch behind them, and the tiles
of the matrix cores with token scales that are not f16 values.  Every output has the bits of the oracle's AVX2 order.  Which way
a product takes is asserted through the library's own functions (C++ symbols; the structures are those of csrc/rmi_internal.h)."""
import ctypes as C

import numpy as np
import pytest

from conftest import bits
from test_gpu_q8_0_x86_gemm import GEMV, T32X32, T64X16, T64X64, plan_of

pytestmark = pytest.mark.gpu

A = 1  # the oracle's AVX2 order


def _activation(hip, oracle, seed, n_tokens, n_in):
    x = hip.synth.activations(seed, n_tokens, n_in)
    per = [oracle.quantize_q8_0(x[t], A) for t in range(n_tokens)]
    return np.stack([p[0] for p in per]), np.stack([p[1] for p in per])


def _run(hip, w, q8, sc, n_out, n_in, r0, r1, stride):
    H, n_tokens = hip.hip, len(q8)
    k = hip.kernel.Q8Kernel(w, n_in, n_out)
    d_q8, d_sc = H.DeviceBuffer.from_array(q8), H.DeviceBuffer.from_array(sc)
    sentinel = np.full((n_tokens, stride), np.float32(-3.75))
    d_y = H.DeviceBuffer.from_array(sentinel)
    H.check(H.lib.rmi_hip_gemv_q8_0_dev(k.w.handle, d_q8.ptr, d_sc.ptr, d_y.ptr, n_tokens, stride, r0, r1, None))
    H.check(H.lib.rmi_hip_synchronize())
    got = d_y.to_array(np.float32, (n_tokens, stride))
    assert np.all(got[:, :r0] == -3.75) and np.all(got[:, r1:] == -3.75), "outside the row range"
    return got[:, r0:r1]


class Groups(C.Structure):
    _fields_ = [("tokens", C.c_uint32), ("groups", C.c_uint32), ("apart", C.c_uint32), ("us", C.c_double)]


def _grouping(hip, n_out, n_in, n_tokens):
    """(whole launch's tokens a group, tokens in a launch of their own, tokens a workgroup takes) of the GEMV."""
    lib, u = hip.hip.lib, C.c_uint32
    lib._Z20rmi_gemv_q8_0_groupsjjj.restype = Groups
    n_oct, n_tiles = (n_in + 255) // 256, (n_out + 7) // 8
    g = lib._Z20rmi_gemv_q8_0_groupsjjj(u(n_oct), u(n_tiles * 8), u(n_tokens))
    waves = -(-n_tiles // lib._Z23rmi_gemv_tiles_per_wavejjj(u(n_oct), u(n_tiles), u(g.tokens)))
    return g.tokens, g.apart, lib._Z27rmi_gemv_q8_0_per_workgroupjjjj(u(waves), u(n_oct), u(g.tokens), u(n_tokens - g.apart))


# The groups that a few rows are spread over are of two and fewer tokens, on the vector ALU, whatever they begin with; five and seven
# tokens of 256 and 1056 columns are one group with its dots on the matrix cores.
@pytest.mark.parametrize("n_in", [256, 1056, 7424, 12288])
@pytest.mark.parametrize("n_tokens", [4, 5, 7, 8, 9, 12, 13, 16, 17, 23, 28, 29])
def test_token_groups(hip, oracle, n_tokens, n_in):
    n_out = 8 * 5 + 3
    w = hip.synth.q8_0_weight(n_in + n_tokens, n_out, n_in)
    q8, sc = _activation(hip, oracle, 60 + n_tokens, n_tokens, n_in)
    for r0, r1, stride in ((0, n_out, n_out), (3, 30, n_out + 5)):
        got = _run(hip, w, q8, sc, n_out, n_in, r0, r1, stride)
        for t in range(n_tokens):
            ref = oracle.matmul_q8_0_quantized(w, q8[t], sc[t], n_in, n_out, A)[r0:r1]
            assert np.array_equal(bits(got[t]), bits(ref)), (t, r0)


def _check_rows(hip, oracle, w, q8, sc, n_out, n_in, ranges):
    for r0, r1, stride in ranges:
        got = _run(hip, w, q8, sc, n_out, n_in, r0, r1, stride)
        rows = np.unique(np.r_[r0:r0 + 16, r1 - 16:r1, np.random.default_rng(r0).integers(r0, r1, 100)])
        wr = np.ascontiguousarray(w.reshape(n_out, -1)[rows]).reshape(-1)
        for t in range(len(q8)):
            assert np.array_equal(bits(got[t, rows - r0]), bits(oracle.matmul_q8_0_quantized(wr, q8[t], sc[t], n_in, rows.size, A))), (t, r0)


# n_out, n_in, tokens, tokens a group, tokens in a launch of their own, tokens a workgroup takes
GROUPED = [
    (4096, 1024, 9, 4, 0, 4), (4096, 1024, 17, 4, 0, 4), (4096, 1056, 13, 8, 0, 4), (2053, 4096, 30, 8, 0, 4), (6144, 2048, 13, 8, 0, 4),  # ragged fours, halves of eights
    (4096, 1024, 23, 8, 0, 8), (4096, 1024, 29, 8, 0, 8), (8003, 2048, 13, 8, 0, 8),  # ragged eights
    (15003, 512, 8, 8, 0, 8), (15003, 2560, 8, 8, 0, 8), (9000, 2560, 8, 8, 0, 4),  # one group of eight, or its halves
    (3003, 12288, 13, 4, 0, 4), (5003, 9984, 10, 4, 0, 4),  # rows too long for eight, ragged fours
    (9603, 7168, 7, 7, 0, 7), (8203, 11776, 5, 4, 1, 4), (8203, 11776, 6, 4, 2, 4), (4003, 11776, 5, 4, 0, 2), (8203, 14080, 5, 4, 1, 4),  # of large matrices: one group; four and the rest
    (515, 14592, 7, 3, 0, 3), (515, 20480, 5, 2, 0, 2)]  # rows too long for four


@pytest.mark.parametrize("n_out,n_in,n_tokens,tokens,apart,per", GROUPED)
def test_groups_of_full_launches(hip, oracle, n_out, n_in, n_tokens, tokens, apart, per):
    assert plan_of(hip.hip, n_out, n_tokens, n_in) == GEMV
    assert _grouping(hip, n_out, n_in, n_tokens) == (tokens, apart, per)
    w = hip.synth.q8_0_weight(n_in + n_tokens, n_out, n_in)
    q8, sc = _activation(hip, oracle, 60 + n_tokens, n_tokens, n_in)
    _check_rows(hip, oracle, w, q8, sc, n_out, n_in, ((0, n_out, n_out), (3, n_out - 2, n_out + 5)))


# sizes of which the estimates once thought too little of the GEMV's time (us by tiles and by groups: the first 45 and 62, the second 78
# and 101, the last 8.8 and 11.1)
@pytest.mark.parametrize("n_out,n_in,n_tokens,tile", [(18626, 2400, 35, T32X32), (13374, 12544, 9, T64X16), (17601, 4576, 37, T32X32),
                                                      (33166, 6144, 17, T32X32), (51481, 6144, 33, T32X32), (9931, 13024, 19, T32X32), (14786, 3840, 10, T64X16),
                                                      (5448, 1120, 30, T32X32)])
def test_products_that_tiles_are_faster_for(hip, n_out, n_in, n_tokens, tile):
    assert plan_of(hip.hip, n_out, n_tokens, n_in) == tile


@pytest.mark.parametrize("n_in,n_tokens", [(1024, 9), (1024, 20), (8192, 5), (8192, 8), (8192, 9)])
def test_large_matrix(hip, oracle, n_tokens, n_in):
    """From 64 M weights on: tiles of 64 x 16 and 32 x 32 for short rows, and for long ones a group of five, two of four and three."""
    n_out = (64 << 20) // n_in + 8
    w = hip.synth.q8_0_weight(3, n_out, n_in)
    q8, sc = _activation(hip, oracle, 90 + n_tokens, n_tokens, n_in)
    _check_rows(hip, oracle, w, q8, sc, n_out, n_in, ((0, n_out, n_out),))


# tiles of 64 x 16, of 32 x 32 and of 64 x 64, each with ragged edges and, but for the first, with blocks beyond whole quads, and the
# GEMV's groups
@pytest.mark.parametrize("n_out,n_in,n_tokens,tile", [(12285, 256, 15, T64X16), (3005, 1056, 20, GEMV), (3005, 1056, 300, T32X32), (4083, 1024, 450, T64X64),
                                                      (4083, 1120, 450, T64X64)])
@pytest.mark.parametrize("odd", [0.1, 1e-40, 70000.0, np.inf, np.nan, -0.0, None])
def test_tiles_and_token_scales(hip, oracle, n_out, n_in, n_tokens, tile, odd):
    """The scale products of a tile come from f16 products of the matrix cores; from a token scale on that is no finite f16 value (a
    caller's own) the vector ALU makes them.  None: nothing but the quantizer's scales, and a weight scale that is
    infinite and one that is subnormal."""
    assert plan_of(hip.hip, n_out, n_tokens, n_in) == tile
    w = hip.synth.q8_0_weight(n_in + 5, n_out, n_in).copy()
    q8, sc = _activation(hip, oracle, 70 + n_tokens, n_tokens, n_in)
    if odd is None:
        scales = w.reshape(n_out, n_in // 32, 34)[:, :, :2].view(np.float16)
        scales[7, 2], scales[9, 1] = np.float16(np.inf), np.float16(3e-7)
    else:
        sc[n_tokens // 2, 3] = odd
        sc[n_tokens - 1, 0] = odd
    got = _run(hip, w, q8, sc, n_out, n_in, 0, n_out, n_out)
    for t in sorted({0, 1, n_tokens // 2 - 1, n_tokens // 2, n_tokens // 2 + 1, n_tokens - 2, n_tokens - 1}):
        ref = oracle.matmul_q8_0_quantized(w, q8[t], sc[t], n_in, n_out, A)
        same = (bits(got[t]) == bits(ref)) | (np.isnan(got[t]) & np.isnan(ref))
        assert np.all(same), (t, np.flatnonzero(~same)[:5])
