"""The forms a linear layer's call may have -- activations of every type, weights that begin anywhere and lie any pitch apart,
results that are columns of a wider tensor, a bias -- at sizes that the streaming tiles and the whole-number GEMM take,
against the CPU oracle."""
import numpy as np
import pytest
import torch

from oracle import gguf_oracle as o
from vllm_gguf_plugin_prism_amd import dispatch as D

pytestmark = pytest.mark.gpu
SIZES = {1: (12, 2080, 4096), 2: (200, 512, 768)}         # route -> rows, N, K


@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("offset,pad,column,spare", [(0, 0, 0, 0), (2, 14, 3, 4), (16, 16, 4, 4), (6, 4, 1, 0)])
@pytest.mark.parametrize("qtype", [o.Q4_K, o.Q5_K, o.Q6_K])
@pytest.mark.parametrize("route", [1, 2])
def test_forms(route, qtype, offset, pad, column, spare, dt):
    from vllm_gguf_plugin_prism_amd import ops
    m, n, k = SIZES[route]
    rng = np.random.default_rng(route + qtype)
    packed = o.make_weights(rng, qtype, n, k)
    rb = packed.shape[1]
    pitch = rb + pad
    assert ops._mmq_route(qtype, n, k, m, pitch) == route
    raw = torch.zeros(offset + n * pitch, dtype=torch.uint8, device="cuda")
    w = raw[offset:].view(n, pitch)[:, :rb]
    w.copy_(torch.from_numpy(packed))
    x = torch.from_numpy(rng.standard_normal((m, k)).astype(np.float32)).to(dt)
    bias = torch.from_numpy(rng.standard_normal(n).astype(np.float32)).to(dt)
    wide = torch.full((m, column + n + spare), 7.0, dtype=dt, device="cuda")
    out = wide[:, column:column + n]
    assert D.fused_mul_mat_gguf(x.cuda(), w, qtype, out=out, bias=bias.cuda()) is out
    want = o.mul_mat_a8(packed, x.float().numpy(), qtype, n, "mmq") + bias.float().numpy()
    # two roundings to 16 bits (product, product plus bias), each half a unit in the last place of 11 or 8 bits
    assert o.rel_l2(out.float().cpu().numpy(), want) <= {torch.float32: 1e-5, torch.float16: 2.0 ** -10, torch.bfloat16: 2.0 ** -7}[dt]
    assert bool((wide[:, :column] == 7).all()) and bool((wide[:, column + n:] == 7).all())
