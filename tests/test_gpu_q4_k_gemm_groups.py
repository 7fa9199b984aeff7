"""The Q4_K prefill GEMM with its rows' super-blocks shared by two or four groups of waves, over 32 and 64 tokens and 128 and 64
rows a workgroup: every plan forced in turn, and the one that is chosen, at rows, tokens and super-blocks around the tiles' edges.
Every output within 1e-4 + 1e-4 |ref| of the AVX2-order result (the tolerance of the kernel's other tests), the integers of every
super-block exact, nothing written beside the results."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# (token tile in units of 32, groups)
_PLANS = [None, ("1", "1"), ("2", "1"), ("1", "2"), ("2", "2"), ("1", "4")]


@pytest.mark.parametrize("n_in", [512, 1024, 1536, 3072])
def test_every_plan_at_the_edges_of_its_tiles(hip, oracle, monkeypatch, n_in):
    H = hip.hip
    for i, (n_tokens, n_out) in enumerate([(16, 1), (31, 63), (32, 64), (33, 65), (64, 127), (65, 129), (97, 200)]):
        w = hip.synth.q4_k_weight(700 + i, n_out, n_in)
        x = hip.synth.activations(720 + i, n_tokens, n_in)
        kernel = hip.kernel.Q4_KKernel(w, n_in, n_out)
        q = [oracle.quantize_row_q8_k(x[t], oracle.AVX2) for t in range(n_tokens)]
        ref = np.zeros((n_tokens, n_out), np.float32)
        for t, (d, qs, bs) in enumerate(q):
            oracle.q4k_forward_prepared(w, d, qs, bs, ref[t], n_in, n_out, 0, 1, oracle.AVX2)
        exact = np.stack([oracle.q4k_q8k_block_ints_matrix(w, n_out, qs, bs) for _, qs, bs in q])
        d_d, d_q, d_b = (H.DeviceBuffer.from_array(np.stack([t[k] for t in q])) for k in range(3))
        d_i = H.DeviceBuffer(exact.size * 4)
        for plan in _PLANS:
            for name, v in zip(("RMI_Q4K_GEMM_TTW", "RMI_Q4K_GEMM_GROUPS"), plan or (None, None)):
                monkeypatch.setenv(name, v) if v else monkeypatch.delenv(name, raising=False)
            out = np.full((n_tokens + 1, n_out), np.nan, np.float32)
            kernel.forward_batched(x, out[:n_tokens], n_in, n_out, matrix_cores=True)
            what = (n_in, n_tokens, n_out, plan)
            assert np.all(np.isnan(out[n_tokens])), what
            assert np.all(np.abs(out[:n_tokens] - ref) <= 1e-4 + 1e-4 * np.abs(ref)), what
            H.check(H.lib.rmi_hip_gemm_block_ints_q4_k_dev(kernel.w.handle, d_d.ptr, d_q.ptr, d_b.ptr, d_i.ptr, n_tokens, None))
            H.check(H.lib.rmi_hip_synchronize())
            assert np.array_equal(d_i.to_array(np.int32, exact.shape), exact), what
        for b in (d_d, d_q, d_b, d_i):
            b.free()
