"""gguf_mmvq_linear_whole: the GEMV without a workspace has the bits of the call with one, or declines and launches nothing."""
import ctypes

import numpy as np
import pytest
import torch

from oracle import gguf_oracle as o

pytestmark = pytest.mark.gpu


# one to four rows, whose quantization the GEMV does itself; a row too long for sixteen waves (K past 32768); five rows; 16 columns more than the result's
@pytest.mark.parametrize("qtype,m,n,k,taken", [(o.Q8_0, 1, 3072, 1024, 1), (o.Q4_K, 2, 37, 256, 1), (o.Q6_K, 3, 64, 4096, 1), (o.IQ2_XXS, 4, 48, 512, 1), (o.Q4_0, 1, 5, 32, 1),
                                               (o.Q4_0, 1, 8, 33024, 0), (o.Q8_0, 4, 8, 40960, 0), (o.Q8_0, 5, 64, 512, 0)])
@pytest.mark.parametrize("dt", (torch.float16, torch.float32))
def test_bits_of_the_call_with_a_workspace(qtype, m, n, k, taken, dt):
    from vllm_gguf_plugin_prism_amd import _lib, ops
    rng = np.random.default_rng(n + k)
    w = torch.from_numpy(o.make_weights(rng, qtype, n, k)).cuda()
    x = torch.from_numpy(rng.standard_normal((m, k)).astype(np.float32)).to(dt).cuda()
    bias = torch.from_numpy(rng.standard_normal(n).astype(np.float32)).to(dt).cuda()
    y, was = torch.full((m, n + 16), 7.0, dtype=dt, device="cuda"), ctypes.c_int(5)
    rc = _lib.lib().gguf_mmvq_linear_whole(w.data_ptr(), w.stride(0), x.data_ptr(), {torch.float32: 0, torch.float16: 1}[dt], y.data_ptr(), n + 16, bias.data_ptr(), int(qtype),
                                           n, k, m, torch.cuda.current_stream().cuda_stream, ctypes.addressof(was))
    assert rc == 0 and was.value == taken and bool((y[:, n:] == 7.0).all())
    if taken:
        assert torch.equal(y[:, :n], ops.ggml_mul_mat_vec_a8(w, x, qtype, n, bias=bias))
    else:
        assert bool((y == 7.0).all())


# rows handed out to half-waves, whose addresses move on by a turn's rows: a last band that is a row short, two turns and twelve, the kernel of eight waves;
# tables of 256 to 2048 entries placed by 1024 threads and by 512
@pytest.mark.parametrize("qtype", (o.IQ2_XXS, o.IQ2_S, o.IQ3_S, o.IQ1_S, o.IQ1_M, o.Q4_0, o.Q8_0))
@pytest.mark.parametrize("n,k", [(2831, 5120), (2555, 3072), (17401, 1024), (100, 512)])
def test_half_waves_and_tables(qtype, n, k):
    from vllm_gguf_plugin_prism_amd import ops
    rng = np.random.default_rng(n)
    w = o.make_weights(rng, qtype, n, k)
    x = rng.standard_normal((1, k)).astype(np.float32)
    rows = np.r_[:12, n // 2:n // 2 + 24, n - 24:n]
    y = ops.ggml_mul_mat_vec_a8(torch.from_numpy(w).cuda(), torch.from_numpy(x).cuda(), qtype, n).cpu().numpy()
    # (fp32 sums of K / 32 block products in another order: 1e-5 of their norm, the tolerance of the GEMV's other tests)
    assert np.isfinite(y).all() and o.rel_l2(y[:, rows], o.mul_mat_a8(w[rows], x, qtype, len(rows), "mmvq")) <= 1e-5
