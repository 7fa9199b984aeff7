"""Attention of a prompt pass through its launch function (a C++ symbol; the structure is that of csrc/attn_prompt.h): which
passes are done in limbs, which blocks of keys and values count as too wide for them, and the same bits as in f64 whatever the
keys, values and queries are.  (test_gpu_prompt_passes.py holds whole passes to single steps, and so to the CPU loop.)"""
import ctypes as C

import numpy as np
import pytest

LAUNCH = "_Z25rmi_launch_attn128_promptPKtS0_S0_jjjjjPfmRK12RmiAttnLimbsbPaS1_iP12ihipStream_t"
IN_LIMBS = "_Z24rmi_attn_prompt_in_limbsjjjRK12RmiAttnLimbsb"
LIMBS_BYTES, LIMBS_AT = "_Z20rmi_attn_limbs_bytesjj", "_Z17rmi_attn_limbs_atPvjj"


class Limbs(C.Structure):
    _fields_ = [("k", C.c_void_p), ("v", C.c_void_p), ("wide", C.c_void_p), ("blocks", C.c_uint32)]


def _in_limbs(lib, heads, step0, n_tok, limbs, hold=True):
    fn = getattr(lib, IN_LIMBS)
    fn.restype = C.c_bool
    return fn(C.c_uint32(heads), C.c_uint32(step0), C.c_uint32(n_tok), C.byref(limbs), C.c_bool(hold))


def test_which_passes_are_done_in_limbs(rmi):
    lib, some = rmi.hip.lib, Limbs(1, 1, 1, 1)  # (only whether there is scratch is looked at)
    assert _in_limbs(lib, 16, 0, 512, some) and not _in_limbs(lib, 16, 0, 360, some)  # 2^20 products of a query and a key
    assert _in_limbs(lib, 16, 1000, 64, some) and not _in_limbs(lib, 16, 1000, 63, some)
    assert not _in_limbs(lib, 16, 0, 512, some, hold=False) and not _in_limbs(lib, 16, 0, 512, Limbs())
    assert _in_limbs(lib, 16, 32768 - 64, 64, some) and not _in_limbs(lib, 16, 32768 - 63, 64, some)  # int32 sums of weighted values


# (whose, position, head, dimension, value): what limbs hold goes up to 127, exclusively
PLANTED = {
    "fits": [("k", 3, 0, 5, 126.9375), ("v", 200, 1, 127, -126.9375), ("q", 100, 2, 0, 126.9375), ("v", 64, 3, 64, 2.0**-24), ("k", 63, 2, 1, -2.0**-24)],
    "key": [("k", 130, 1, 77, 127.0)],
    "value": [("v", 0, 2, 0, -127.0), ("v", -1, 0, 127, 4000.0)],
    "value of two heads": [("v", 65, 0, 3, 65504.0), ("v", 127, 3, 3, 128.0)],
    "query of a tile's first half": [("q", 32, 5, 9, 127.0)],
    "query of a tile's second half": [("q", -1, 0, 120, -300.0)],
    "not finite": [("v", 300, 1, 4, np.inf), ("k", 310, 2, 4, -np.inf), ("q", 40, 7, 4, np.nan), ("v", 330, 3, 0, np.nan)],
}


@pytest.mark.gpu
@pytest.mark.parametrize("heads,kv_heads,step0,n_tok,one_launch", [
    (8, 4, 300, 320, True), (8, 4, 293, 321, False), (8, 4, 0, 528, True), (16, 4, 333, 160, True), (8, 4, 1000, 143, False), (8, 4, 129, 433, True), (64, 8, 200, 161, True)])
@pytest.mark.parametrize("planted", PLANTED)
def test_limbs_have_the_bits_of_f64(hip, heads, kv_heads, step0, n_tok, one_launch, planted):
    """Passes of whole tiles and of a rest of 1, 15, 16 and 17 positions; in one launch, and with scratch for a tile at a time;
    more tiles than compute units (64 heads), where one workgroup does all 32 positions that limbs don't hold, and fewer, where
    two do."""
    H = hip.hip
    rng = np.random.default_rng(n_tok)
    n_keys, n_blocks = step0 + n_tok, (step0 + n_tok + 63) // 64
    host = {"q": rng.standard_normal((n_tok, heads, 128)) * 3, "k": rng.standard_normal((n_keys, kv_heads, 128)) * 3, "v": rng.standard_normal((n_keys, kv_heads, 128))}
    host = {name: a.astype(np.float16) for name, a in host.items()}
    wide = np.zeros((2, kv_heads, n_blocks), np.uint32)
    for name, t, head, dim, value in PLANTED[planted]:
        host[name][t, head, dim] = value
        if name != "q" and not abs(value) < 127:
            wide["kv".index(name), head, t % n_keys // 64] = 1
    dev = {name: H.DeviceBuffer.from_array(a) for name, a in host.items()}
    stride = (n_keys + 127) // 128 * 128
    floats = heads * 32 * stride * ((n_tok + 31) // 32 if one_launch else 1)
    scratch = H.DeviceBuffer(floats * 4)
    size, at = getattr(H.lib, LIMBS_BYTES), getattr(H.lib, LIMBS_AT)
    size.restype, at.restype = C.c_size_t, Limbs
    limb_bytes = size(C.c_uint32(kv_heads), C.c_uint32(n_keys))
    assert limb_bytes == 2 * kv_heads * n_blocks * (64 * 128 * 4 + 4)
    limb_buf = H.DeviceBuffer(limb_bytes)
    results = []
    for limbs in (at(C.c_void_p(limb_buf.ptr), C.c_uint32(kv_heads), C.c_uint32(n_keys)), Limbs()):
        assert _in_limbs(H.lib, heads, step0, n_tok, limbs) == bool(limbs.blocks)
        q8, scales = H.DeviceBuffer(n_tok * heads * 128), H.DeviceBuffer(n_tok * heads * 4 * 4)
        assert getattr(H.lib, LAUNCH)(C.c_void_p(dev["q"].ptr), C.c_void_p(dev["k"].ptr), C.c_void_p(dev["v"].ptr), C.c_uint32(step0), C.c_uint32(n_tok),
                                      C.c_uint32(kv_heads * 128), C.c_uint32(heads), C.c_uint32(kv_heads), C.c_void_p(scratch.ptr), C.c_size_t(floats),
                                      C.byref(limbs), C.c_bool(True), C.c_void_p(q8.ptr), C.c_void_p(scales.ptr), C.c_int(H.ROUND_TIES_EVEN), None) == 0
        H.check(H.lib.rmi_hip_synchronize())
        if limbs.blocks:
            flags = np.empty((2, kv_heads, n_blocks), np.uint32)
            H.check(H.lib.rmi_hip_memcpy_d2h(flags.ctypes.data, limbs.wide, flags.nbytes))
            assert np.array_equal(flags, wide)
        results.append((q8.to_array(np.int8, (n_tok, heads, 128)), scales.to_array(np.uint32, (n_tok, heads, 4))))
    assert np.array_equal(results[0][0], results[1][0]) and np.array_equal(results[0][1], results[1][1])
