"""Q8_0 products of more than eight tokens in the x86-64 order: every token's bits are those of the eight-token GEMV (held to the
oracle by test_gpu_q8_0.py) and, for some tokens, of the restated AVX2 kernel itself.  Through the public entry, which takes
tiles of the matrix cores or the GEMV's token groups as its estimates say, and tile by tile through the library's own launch
function (a C++ symbol; the structures are those of csrc/rmi_internal.h), whatever the estimates say."""
import ctypes as C
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

GEMV, T64X64, T32X32, T64X16 = range(4)


class Weight(C.Structure):
    _fields_ = [(n, C.c_uint32) for n in ("dtype", "n_in", "n_out", "n_tiles", "n_units")] + [
        ("tile_bytes", C.c_size_t), ("nbytes", C.c_size_t), ("data", C.c_void_p)]


class Problem(C.Structure):
    _fields_ = [(n, C.c_void_p) for n in ("w", "x_q8", "x_scales", "y")] + [
        (n, C.c_uint32) for n in ("n_in", "n_oct", "y_stride", "row_start", "row_end", "tile0", "n_tiles", "n_tokens")]


def plan_of(H, n_rows, tokens, n_in):
    return H.lib._Z22rmi_gemm_q8_0_x86_planjjj(C.c_uint32((n_rows + 7) // 8 * 8), C.c_uint32(tokens), C.c_uint32(n_in))


def _tiled(H, tile, weight, q, s, n_out, stride, first, last):
    """The rows [first, last) of a product in tiles of one size."""
    tokens, n_in = q.shape
    w = C.cast(weight.w.handle, C.POINTER(Weight)).contents
    assert (w.n_in, w.n_out, w.nbytes) == (n_in, n_out, w.n_tiles * w.tile_bytes)
    d_q, d_s = H.DeviceBuffer.from_array(q), H.DeviceBuffer.from_array(s)
    d_y = H.DeviceBuffer.from_array(np.full((tokens, stride), -7.0, np.float32))
    p = Problem(w.data, d_q.ptr, d_s.ptr, d_y.ptr, n_in, w.n_units, stride, first, last, first // 8, (last + 7) // 8 - first // 8, 0)
    assert H.lib._Z24rmi_launch_gemm_q8_0_x8610RmiX86PlanRK14RmiGemvProblemjP12ihipStream_t(C.c_int(tile), C.byref(p), C.c_uint32(tokens), None) == 0
    H.check(H.lib.rmi_hip_synchronize())
    y = d_y.to_array(np.float32, (tokens, stride))
    for b in (d_q, d_s, d_y):
        b.free()
    return y


def _same(a, b):
    return ((a.view(np.uint32) == b.view(np.uint32)) | (np.isnan(a) & np.isnan(b))).all()


def _run(H, weight, q, s, n_out, stride, first, last):
    tokens, n_in = q.shape
    d_q, d_s = H.DeviceBuffer.from_array(q), H.DeviceBuffer.from_array(s)
    d_y = H.DeviceBuffer.from_array(np.full((tokens, stride), -7.0, np.float32))
    out = []
    for group in (tokens, 8):  # the whole batch in one call, and eight at a time through the GEMV
        for t in range(0, tokens, group):
            n = min(group, tokens - t)
            H.check(H.lib.rmi_hip_gemv_q8_0_dev(weight.w.handle, d_q.ptr + t * n_in, d_s.ptr + t * (n_in // 32) * 4, d_y.ptr + t * stride * 4, n, stride,
                                                first, last, None))
        H.check(H.lib.rmi_hip_synchronize())
        out.append(d_y.to_array(np.float32, (tokens, stride)))
    for b in (d_q, d_s, d_y):
        b.free()
    return out


@pytest.mark.parametrize("n_in,n_out,tokens", [
    (32, 40, 9), (96, 8200, 640), (288, 4111, 512), (1024, 1000, 200), (1440, 333, 13), (992, 130, 33), (256, 70000, 16), (256, 70003, 12),
    (2048, 1024, 512), (3072, 64, 65), (160, 17, 300)])
def test_batches_have_the_bits_of_the_gemv(hip, oracle, n_in, n_out, tokens):
    H = hip.hip
    rng = np.random.default_rng(n_in + n_out + tokens)
    w = hip.synth.q8_0_weight(n_out, n_out, n_in)
    kernel = hip.kernel.Q8Kernel(w, n_in, n_out)
    q = rng.integers(-128, 128, (tokens, n_in), dtype=np.int8)
    s = rng.uniform(0, 2, (tokens, n_in // 32)).astype(np.float32)
    whole, eights = _run(H, kernel, q, s, n_out, n_out, 0, n_out)
    assert np.array_equal(whole.view(np.uint32), eights.view(np.uint32))
    for t in (0, tokens // 2, tokens - 1):
        qt = np.maximum(q[t], -127)  # (the restated kernel is the reference's, which is wrong for quants of -128)
        ref = oracle.matmul_q8_0_quantized(w, qt.view(np.uint8), s[t], n_in, n_out, oracle.AVX2)
        y = np.zeros(n_out, np.float32)
        kernel.forward_prequantized(qt.view(np.uint8), s[t], y, n_in, n_out, 0, 1)
        assert np.array_equal(y.view(np.uint32), ref.view(np.uint32))
        if (q[t] >= -127).all():
            assert np.array_equal(whole[t].view(np.uint32), ref.view(np.uint32))


@pytest.mark.parametrize("first,last,stride", [(0, 1000, 1003), (3, 997, 1000), (8, 9, 1000), (61, 130, 131), (992, 1000, 1001)])
def test_row_ranges_and_strides(hip, first, last, stride):
    """Rows outside the range keep what was there; token strides that are no multiple of sixteen bytes."""
    rng = np.random.default_rng(first)
    kernel = hip.kernel.Q8Kernel(hip.synth.q8_0_weight(5, 1000, 352), 352, 1000)
    q, s = rng.integers(-127, 128, (150, 352), dtype=np.int8), rng.uniform(0, 2, (150, 11)).astype(np.float32)
    whole, eights = _run(hip.hip, kernel, q, s, 1000, stride, first, last)
    assert np.array_equal(whole.view(np.uint32), eights.view(np.uint32))
    outside = np.ones(stride, bool)
    outside[first:last] = False
    assert (whole[:, outside] == -7.0).all()


def test_special_scales(hip):
    """Zero, subnormal, huge, infinite and NaN scales of either operand."""
    rng = np.random.default_rng(1)
    n_in, n_out, tokens = 320, 200, 130
    w = hip.synth.q8_0_weight(3, n_out, n_in).reshape(-1, 34)
    special = np.array([0x0000, 0x8000, 0x0001, 0x7bff, 0x7c00, 0xfc00, 0x7e00], np.uint16)
    at = rng.choice(w.shape[0], 60, replace=False)
    w[at, :2] = special[rng.integers(0, special.size, 60)].view(np.uint8).reshape(60, 2)
    kernel = hip.kernel.Q8Kernel(w.reshape(-1), n_in, n_out)
    q, s = rng.integers(-127, 128, (tokens, n_in), dtype=np.int8), rng.uniform(0, 2, (tokens, 10)).astype(np.float32)
    s[rng.integers(0, tokens, 40), rng.integers(0, 10, 40)] = rng.choice(np.array([0.0, -0.0, 1e-40, 3e38, np.inf, -np.inf, np.nan], np.float32), 40)
    q[7] = 0
    whole, eights = _run(hip.hip, kernel, q, s, n_out, n_out, 0, n_out)
    nan = np.isnan(eights)
    assert np.array_equal(np.isnan(whole), nan)
    assert np.array_equal(whole.view(np.uint32)[~nan], eights.view(np.uint32)[~nan])


# tiles of 32 x 32, of 64 x 64 and of 64 x 16, eight whole quads of blocks and one block
@pytest.mark.parametrize("n_out,n_in,tokens", [(3005, 1056, 300), (4083, 1056, 450), (20003, 1056, 12)])
def test_a_scale_that_is_no_f16_value_at_any_block(hip, n_out, n_in, tokens):
    """Scales are f16 values, as the quantizer leaves them, but for one: in the first quad, at both ends of inner ones, in the last
    and in the block behind them.  The quads in front of it take the other way."""
    rng = np.random.default_rng(n_out)
    kernel = hip.kernel.Q8Kernel(hip.synth.q8_0_weight(9, n_out, n_in), n_in, n_out)
    q = rng.integers(-127, 128, (tokens, n_in), dtype=np.int8)
    f16 = rng.uniform(0, 2, (tokens, n_in // 32)).astype(np.float16).astype(np.float32)
    for block in (None, 0, 3, 4, 11, 20, 31, 32):
        s = f16.copy()
        if block is not None:
            s[tokens * 2 // 3, block] = 0.1
        whole, eights = _run(hip.hip, kernel, q, s, n_out, n_out, 0, n_out)
        assert np.array_equal(whole.view(np.uint32), eights.view(np.uint32)), block


def test_any_token_scale_takes_about_as_long(hip):
    """Scales that are f16 values and others: the same work but for one vector instruction in ten (measured 1.03; 2 is far from
    both that and a second, slower pass over the tile, which took 14 times as long)."""
    H, (n_out, n_in, tokens) = hip.hip, (4096, 1024, 512)
    rng = np.random.default_rng(4)
    kernel = hip.kernel.Q8Kernel(hip.synth.q8_0_weight(2, n_out, n_in), n_in, n_out)
    d_q = H.DeviceBuffer.from_array(rng.integers(-127, 128, (tokens, n_in), dtype=np.int8))
    d_y = H.DeviceBuffer(tokens * n_out * 4)
    scales = rng.uniform(0.5, 1, (tokens, n_in // 32)).astype(np.float16).astype(np.float32)
    best = []
    for s in (scales, scales * np.float32(1.0001)):
        d_s, times = H.DeviceBuffer.from_array(s), []
        for _ in range(5):
            H.check(H.lib.rmi_hip_synchronize())
            t0 = time.perf_counter()
            for _ in range(50):
                H.check(H.lib.rmi_hip_gemv_q8_0_dev(kernel.w.handle, d_q.ptr, d_s.ptr, d_y.ptr, tokens, n_out, 0, n_out, None))
            H.check(H.lib.rmi_hip_synchronize())
            times.append(time.perf_counter() - t0)
        best.append(min(times))
    assert best[1] < 2 * best[0], best


SIZES = {T64X64: 150, T32X32: 75, T64X16: 37}  # tokens: two whole tiles and a ragged one


# quads of four blocks and blocks behind them: 0 + 3, 1 + 1, 7 + 3, 8 + 0, 8 + 1, 8 + 2
@pytest.mark.parametrize("n_in", [96, 160, 992, 1024, 1056, 1088])
@pytest.mark.parametrize("tile", SIZES)
def test_every_tile(hip, oracle, tile, n_in):
    """Zero, subnormal and large token scales that are f16 values, then one that is none in the first, an inner and the last block."""
    n_out, tokens, nb = 203, SIZES[tile], n_in // 32
    rng = np.random.default_rng(n_in + tile)
    w = hip.synth.q8_0_weight(n_in, n_out, n_in)
    kernel = hip.kernel.Q8Kernel(w, n_in, n_out)
    q = rng.integers(-127, 128, (tokens, n_in), dtype=np.int8)
    f16 = rng.uniform(0, 2, (tokens, nb)).astype(np.float16)
    f16[rng.integers(0, tokens, 40), rng.integers(0, nb, 40)] = rng.choice(np.array([0.0, -0.0, 6e-8, 3e-7, 6e-5, -5e-6, 65504.0], np.float16), 40)
    for block in [None, 0, nb // 2, nb - 1]:
        s = f16.astype(np.float32)
        if block is not None:
            s[tokens // 2, block] = 0.1
        got, eights = _tiled(hip.hip, tile, kernel, q, s, n_out, n_out, 0, n_out), _run(hip.hip, kernel, q, s, n_out, n_out, 0, n_out)[1]
        assert np.array_equal(got.view(np.uint32), eights.view(np.uint32)), block
        for t in (0, tokens // 2, tokens - 1):
            ref = oracle.matmul_q8_0_quantized(w, q[t].view(np.uint8), s[t], n_in, n_out, oracle.AVX2)
            assert np.array_equal(got[t].view(np.uint32), ref.view(np.uint32)), (block, t)


@pytest.mark.parametrize("f16", [True, False])
@pytest.mark.parametrize("tile", SIZES)
def test_row_ranges_and_strides_of_every_tile(hip, tile, f16):
    rng = np.random.default_rng(tile)
    kernel = hip.kernel.Q8Kernel(hip.synth.q8_0_weight(5, 1000, 352), 352, 1000)
    tokens = SIZES[tile]
    q, s = rng.integers(-127, 128, (tokens, 352), dtype=np.int8), rng.uniform(0, 2, (tokens, 11)).astype(np.float16 if f16 else np.float32).astype(np.float32)
    for first, last, stride in ((0, 1000, 1003), (3, 997, 1000), (8, 9, 1000), (61, 130, 131), (992, 1000, 1001)):
        got, eights = _tiled(hip.hip, tile, kernel, q, s, 1000, stride, first, last), _run(hip.hip, kernel, q, s, 1000, stride, first, last)[1]
        assert np.array_equal(got.view(np.uint32), eights.view(np.uint32)), (first, last)
        outside = np.ones(stride, bool)
        outside[first:last] = False
        assert (got[:, outside] == -7.0).all()


@pytest.mark.parametrize("f16", [True, False])
@pytest.mark.parametrize("tile", SIZES)
def test_special_scales_of_every_tile(hip, tile, f16):
    """Zero, subnormal, largest, infinite and NaN weight scales; token scales of all kinds that f16 holds, or that f32 does."""
    rng = np.random.default_rng(tile)
    n_in, n_out, tokens = 352, 200, SIZES[tile]
    w = hip.synth.q8_0_weight(3, n_out, n_in).reshape(-1, 34)
    special = np.array([0x0000, 0x8000, 0x0001, 0x83ff, 0x7bff, 0x7c00, 0xfc00, 0x7e00], np.uint16)
    at = rng.choice(w.shape[0], 60, replace=False)
    w[at, :2] = special[rng.integers(0, special.size, 60)].view(np.uint8).reshape(60, 2)
    kernel = hip.kernel.Q8Kernel(w.reshape(-1), n_in, n_out)
    q, s = rng.integers(-127, 128, (tokens, n_in), dtype=np.int8), rng.uniform(0, 2, (tokens, 11)).astype(np.float16).astype(np.float32)
    odd = [0.0, -0.0, 6e-8, 6e-5, 65504.0] if f16 else [0.0, -0.0, 1e-40, 70000.0, 3e38, np.inf, -np.inf, np.nan]
    s[rng.integers(0, tokens, 40), rng.integers(0, 11, 40)] = rng.choice(np.array(odd, np.float16 if f16 else np.float32), 40).astype(np.float32)
    q[7] = 0
    assert _same(_tiled(hip.hip, tile, kernel, q, s, n_out, n_out, 0, n_out), _run(hip.hip, kernel, q, s, n_out, n_out, 0, n_out)[1])


@pytest.mark.parametrize("n_out,n_in,tokens,tile", [(6144, 1024, 1024, T64X64), (4083, 1056, 450, T64X64), (1024, 3072, 512, T32X32), (3005, 1056, 300, T32X32),
                                                    (20003, 1056, 12, T64X16), (6144, 2048, 13, GEMV), (3005, 1056, 20, GEMV), (151936, 1024, 8, GEMV)])
def test_what_the_public_entry_takes(hip, n_out, n_in, tokens, tile):
    """On 256 compute units; other tests that name a tile by a product's size rest on this."""
    assert plan_of(hip.hip, n_out, tokens, n_in) == tile
