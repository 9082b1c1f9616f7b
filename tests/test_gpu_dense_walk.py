"""The walking codebook GEMM (csrc/dense_walk_core.h) at the edges of its tiles and panels, in the forms that a linear layer's call may have, and the kernel
behind it where that still runs, against the dequantized weights multiplied in float64."""
import numpy as np
import pytest
import torch

from vllm_gguf_plugin_prism_amd import _lib, dispatch as D, synth

pytestmark = pytest.mark.gpu
FORMATS = sorted(D.IMATRIX_QUANT_TYPES)
TOLERANCE = {torch.float16: 2.0 ** -10, torch.bfloat16: 2.0 ** -7}   # two roundings to 16 bits (product, product plus bias), each half a unit in the last place of 11 or 8 bits


EDGES = [(33, 4155, 512, 2, (1, 4)), (68, 4327, 1280, 0, (1, 4)), (69, 4313, 2304, 6, (1, 4)), (35, 1144, 512, 0, (1, 8)), (71, 1215, 3072, 4, (1, 8)), (79, 1564, 5120, 0, (1, 8)),
         (65, 5539, 768, 0, (2, 4)), (99, 4120, 1280, 8, (2, 4)), (65, 5513, 2304, 0, (2, 4)), (553, 466, 768, 10, (2, 8)), (35, 4405, 2304, 0, (2, 8)), (68, 2981, 4352, 2, (2, 8)),
         (129, 6575, 768, 12, (3, 4)), (197, 4104, 1280, 0, (3, 4)), (135, 5986, 2304, 0, (3, 4)), (203, 4894, 768, 0, (4, 4)), (193, 5530, 1280, 14, (4, 4)), (203, 5506, 2304, 0, (4, 4)),
         (614, 1380, 1536, 0, (4, 8)), (613, 915, 2304, 2, (4, 8)), (194, 2856, 5120, 0, (4, 8)),
         (5, 41, 1280, 0, (17, 8)), (16, 1182, 2304, 2, (17, 8)), (32, 3001, 1280, 6, (17, 8)), (5, 1801, 5120, 0, (17, 8)), (5, 8254, 512, 4, (17, 4)), (9, 11006, 1280, 0, (17, 4)),
         (13, 24757, 2304, 0, (17, 4))]   # (17: one tile of rows, loaded as they lie)
BEHIND = [(D.IQ3_XXS, 4, 230, 1280), (D.IQ3_XXS, 71, 210, 1536), (D.IQ3_XXS, 129, 210, 1280), (D.IQ3_XXS, 35, 8986, 512), (D.IQ4_XS, 66, 5487, 512), (D.IQ3_XXS, 129, 3343, 512),
          (D.IQ2_S, 24, 4096, 18944), (D.IQ1_S, 65, 300, 2816), (D.IQ2_S, 1025, 300, 512)]


def plan(qt, m, n, k, pitch, size=None):
    L = _lib.lib()
    return divmod(L.gguf_dense_linear_walk(int(qt), n, k, m, pitch, L.gguf_dense_linear_workspace_bytes(n, k, m) if size is None else size), 16)


def check(qt, dt, m, n, k, want_plan, pad=0, offset=0, column=0, spare=0, size=None):
    from vllm_gguf_plugin_prism_amd import ops
    rng = np.random.default_rng(m + n + k)
    packed = torch.from_numpy(synth.make_weights(rng, qt, n, k)).cuda()
    rb = packed.shape[1]
    w = torch.zeros(offset + n * (rb + pad), dtype=torch.uint8, device="cuda")[offset:].view(n, rb + pad)[:, :rb]
    w.copy_(packed)
    got = plan(qt, m, n, k, rb + pad, size)
    assert got == want_plan if want_plan is not None else got[0]
    x = torch.from_numpy(rng.standard_normal((m, k)).astype(np.float32) + 0.3).to(dt).cuda()
    bias = torch.from_numpy(rng.standard_normal(n).astype(np.float32)).to(dt).cuda()
    wide = torch.full((m, column + n + spare), 7.0, dtype=dt, device="cuda")
    out = wide[:, column:column + n]
    if size is None:
        assert ops.dense_linear(w, x, qt, n, out=out, bias=bias) is out
    else:
        ws = torch.empty(size, dtype=torch.uint8, device="cuda")
        _lib.check(_lib.lib().gguf_dense_linear(w.data_ptr(), rb + pad, x.data_ptr(), 1 if dt == torch.float16 else 2, ws.data_ptr(), out.data_ptr(), out.stride(0), bias.data_ptr(),
                                                int(qt), n, k, m, size, torch.cuda.current_stream().cuda_stream), "gguf_dense_linear")
    want = x.double() @ ops.ggml_dequantize(packed, qt, n, k, dt).double().T + bias.double()
    assert ((out.double() - want).norm() / want.norm()).item() <= TOLERANCE[dt]
    assert bool((wide[:, :column] == 7).all()) and bool((wide[:, column + n:] == 7).all())


# each height of tiles with each number of waves that it has: waves without a panel, with one, two and three; last tiles of rows and columns in part; rows of W a
# pitch apart that moves them through the positions inside 16 bytes
@pytest.mark.parametrize("qt", FORMATS)
@pytest.mark.parametrize("m,n,k,pad,want", EDGES)
def test_edges(qt, m, n, k, pad, want):
    check(qt, torch.bfloat16, m, n, k, want, pad)


# K in blocks of 32: the last panel has one block, three, seven
@pytest.mark.parametrize("m,n,k,pad", [(70, 4100, 2080, 0), (45, 3333, 1120, 2), (130, 4444, 2528, 0), (37, 3333, 992, 6), (20, 3333, 160, 0), (32, 1700, 992, 2), (7, 2001, 2080, 0)])
def test_last_panels(m, n, k, pad):
    check(D.IQ4_NL, torch.float16, m, n, k, None, pad)


# both types, weights that begin anywhere, results that are columns of a wider tensor
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("offset,pad,column,spare", [(0, 0, 0, 0), (2, 14, 3, 4), (16, 16, 4, 4), (6, 4, 1, 0)])
@pytest.mark.parametrize("m", [34, 13])
@pytest.mark.parametrize("qt", FORMATS)
def test_forms(qt, m, offset, pad, column, spare, dt):
    check(qt, dt, m, 3301, 1280, None, pad, offset, column, spare)


# a value that is not a number stays in its row
@pytest.mark.parametrize("m", [34, 13])
def test_rows_do_not_meet(m):
    from vllm_gguf_plugin_prism_amd import ops
    n, k = 3301, 1280
    w = torch.from_numpy(synth.make_weights(np.random.default_rng(1), D.IQ3_S, n, k)).cuda()
    assert plan(D.IQ3_S, m, n, k, w.shape[1])[0]
    x = torch.randn(m, k, dtype=torch.bfloat16, device="cuda")
    y = ops.dense_linear(w, x, D.IQ3_S, n)
    x[m - 1, 1000] = float("nan")
    z = ops.dense_linear(w, x, D.IQ3_S, n)
    assert bool(z[m - 1].isnan().all()) and torch.equal(z[:m - 1], y[:m - 1])


# the kernel behind it: products that it does not take, and a workspace with no room for the rows
@pytest.mark.parametrize("qt,m,n,k", BEHIND)
def test_the_kernel_behind_it(qt, m, n, k):
    check(qt, torch.float16, m, n, k, (0, 0))


@pytest.mark.parametrize("qt", [D.IQ4_XS, D.IQ1_M, D.IQ4_NL])
def test_a_workspace_without_room(qt):
    m, n, k = 255, 5120, 1024
    size = -(-m // 32) * k // 256 * 16384
    assert _lib.lib().gguf_dense_linear_workspace_bytes(n, k, m) == size   # (as much as the rows take: the partial tiles take less)
    check(qt, torch.bfloat16, m, n, k, (0, 0), size=size - 16)


# captured once, replayed on other activations with eager work in between
def test_replays_as_eager():
    m, n, k = 40, 4096, 4096
    w = torch.from_numpy(synth.make_weights(np.random.default_rng(3), D.IQ4_XS, n, k)).cuda()
    assert plan(D.IQ4_XS, m, n, k, w.shape[1])[0]
    xs = [torch.randn(m, k, dtype=torch.bfloat16, device="cuda") for _ in range(4)]
    x = xs[0].clone()
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        D.fused_mul_mat_gguf(x, w, D.IQ4_XS)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = D.fused_mul_mat_gguf(x, w, D.IQ4_XS)
    for xi in xs:
        x.copy_(xi)
        eager = D.fused_mul_mat_gguf(x, w, D.IQ4_XS).clone()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager)
