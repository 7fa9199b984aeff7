"""Products of several tokens in the x86-64 order (matmul_q8_0_vs_q8_0_avx2, src/ops/kernel/q8_0/avx2.rs:71-173): the GEMV's
token groups, of eight and of four, whole, ragged (the last group begins earlier) and with a launch behind them, and the tiles
of the matrix cores with token scales that are not f16 values.  Every output has the bits of the oracle's AVX2 order."""
import numpy as np
import pytest

from conftest import bits

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


# rows of 1024 and 1056 columns are staged by eights, 7424 and 12288 by fours; 9..12 and 17..20 tokens go by fours on any row
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


@pytest.mark.parametrize("n_in,n_tokens", [(1024, 9), (1024, 20), (8192, 5), (8192, 8), (8192, 9)])
def test_large_matrix(hip, oracle, n_tokens, n_in):
    """From 64 M weights on the tokens beyond whole groups are a launch of their own, and long rows take larger groups."""
    n_out = (64 << 20) // n_in + 8
    w = hip.synth.q8_0_weight(3, n_out, n_in)
    q8, sc = _activation(hip, oracle, 90 + n_tokens, n_tokens, n_in)
    got = _run(hip, w, q8, sc, n_out, n_in, 0, n_out, n_out)
    rows = np.unique(np.concatenate([np.arange(16), np.arange(n_out - 16, n_out), np.random.default_rng(1).integers(0, n_out, 200)]))
    wr = np.ascontiguousarray(w.reshape(n_out, -1)[rows]).reshape(-1)
    for t in range(n_tokens):
        assert np.array_equal(bits(got[t, rows]), bits(oracle.matmul_q8_0_quantized(wr, q8[t], sc[t], n_in, rows.size, A))), t


# tiles of 64 x 16, of 32 x 32 and of 64 x 64, each with ragged edges, one of them with blocks beyond whole quads
@pytest.mark.parametrize("n_out,n_in,n_tokens", [(12285, 256, 15), (3005, 1056, 75), (4083, 1024, 450)])
@pytest.mark.parametrize("odd", [0.1, 1e-40, 70000.0, np.inf, np.nan, -0.0, None])
def test_tiles_and_token_scales(hip, oracle, n_out, n_in, n_tokens, odd):
    """The scale products of a tile come from f16 products of the matrix cores; a token scale that is no finite f16 value (a
    caller's own) sends its tile to the vector ALU.  None: nothing but the quantizer's scales, and a weight scale that is
    infinite and one that is subnormal."""
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
