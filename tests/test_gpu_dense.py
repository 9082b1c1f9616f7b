"""The codebook formats' GEMM (csrc/dense_core.h; sizes that the walking waves of csrc/dense_walk_core.h do not take) at the edges of its tiles, of the runs its workgroups share and of K, with
padded rows, a column slice for the result and a bias, against the dequantized weights multiplied in float64."""
import numpy as np
import pytest
import torch

from vllm_gguf_plugin_prism_amd import dispatch as D
from vllm_gguf_plugin_prism_amd import synth

pytestmark = pytest.mark.gpu
FORMATS = sorted(D.IMATRIX_QUANT_TYPES)


def _check(qt, dt, m, n, k, pad=0, seed=0):
    from vllm_gguf_plugin_prism_amd import _lib, ops
    L = _lib.lib()
    rng = np.random.default_rng(seed + m + n + k)
    packed = torch.from_numpy(synth.make_weights(rng, qt, n, k)).cuda()
    assert L.gguf_dense_linear_walk(int(qt), n, k, m, packed.shape[1] + pad, L.gguf_dense_linear_workspace_bytes(n, k, m)) == 0
    w = torch.zeros(n, packed.shape[1] + pad, dtype=torch.uint8, device="cuda")[:, :packed.shape[1]]
    w.copy_(packed)
    x = torch.from_numpy(rng.standard_normal((m, k)).astype(np.float32)).to(dt).cuda()
    bias = torch.from_numpy(rng.standard_normal(n).astype(np.float32)).to(dt).cuda()
    merged = torch.full((m, n + 5), 7.0, dtype=dt, device="cuda")
    assert ops.dense_linear(w, x, qt, n, out=merged[:, 3:n + 3], bias=bias) is not None, "not served"
    want = x.double() @ ops.ggml_dequantize(packed, qt, n, k, dt).double().T + bias.double()
    got = merged[:, 3:n + 3].double()
    assert ((got - want).norm() / want.norm()).item() <= (6e-4 if dt == torch.float16 else 5e-3)
    assert bool((merged[:, :3] == 7).all()) and bool((merged[:, n + 3:] == 7).all())
    assert torch.equal(D.fused_mul_mat_gguf(x, w, qt, bias=bias), merged[:, 3:n + 3].contiguous())   # (stores of four values)


# every format: one row over a tile of 128 weight rows, part of a tile of 64 rows of X
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("qt", FORMATS)
def test_formats(qt, dt):
    _check(qt, dt, 1057, 129, 768)


# tiles of 64, 128 and 256 rows, one row over and under; one unit of K; runs that begin and end inside tiles
@pytest.mark.parametrize("m,n,k,pad", [(1041, 1, 256, 0), (64, 640, 1280, 2), (65, 300, 2816, 0), (129, 8200, 512, 6), (255, 250, 2560, 0),
                                       (257, 201, 2304, 4), (384, 6000, 512, 0)])
def test_tile_edges(m, n, k, pad):
    _check(D.IQ4_XS, torch.bfloat16, m, n, k, pad)


# K in blocks of 32: half a step at the end, parts of a unit
@pytest.mark.parametrize("m,k", [(70, 32), (70, 64), (70, 96), (1070, 288), (1070, 480), (70, 2080)])
def test_ragged_k(m, k):
    _check(D.IQ4_NL, torch.float16, m, 260, k)
