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
