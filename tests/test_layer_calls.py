"""The compiled layer calls (csrc/torch_binding/gguf_calls.cpp): the path they pick is dispatch.py's, what they do not
serve falls back to Python, and their results are those of the Python path bit for bit."""
import numpy as np
import pytest
import torch

from vllm_gguf_plugin_prism_amd import dispatch as D
from vllm_gguf_plugin_prism_amd import synth


def test_path_is_the_one_of_dispatch():
    calls = D._calls()
    assert calls is not D._NoCalls, "build the package first"
    for qt in (t for t in range(-2, 34) if t != D.Q8_1):     # (no kernel takes Q8_1)
        for batch in (0, 1, 2, 3, 6, 7, 8, 9, 16, 17, 4096):
            for rows in (1, 5120, 5121, 20000):
                try:
                    want = D.select_mul_mat_path(qt, batch, rows)
                except NotImplementedError:
                    want = None
                assert calls.mul_mat_path(qt, batch, rows) == (want if want in ("mmvq", "mmq") else None)


def test_calls_decline_what_they_do_not_serve():
    calls, w, x = D._calls(), torch.zeros(8, 18, dtype=torch.uint8), torch.zeros(1, 32)
    assert calls.linear(x, w, D.Q4_0, None, None) is None          # not on a GPU
    assert calls.linear("x", w, D.Q4_0, None, None) is None
    assert calls.merged_linear(x, w, ["q"], {}, [D.Q4_0], None) is None
    assert calls.embedding(x, w, D.Q4_0, 32, torch.float16) is None
    with pytest.raises(TypeError):
        calls.linear(x)


def _both(monkeypatch, fn):
    got = fn()
    with monkeypatch.context() as m:
        m.setattr(D, "_CALLS", D._NoCalls)
        want = fn()
    torch.cuda.synchronize()
    assert got.shape == want.shape and got.dtype == want.dtype and torch.equal(got, want)


@pytest.mark.gpu
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("m", [1, 6, 7, 40])
def test_results_are_those_of_the_python_path(m, dt, monkeypatch):
    rng = np.random.default_rng(m)
    k, e, inner, top_k = 512, 8, 256, 2

    def packed(qt, n, kk):
        return torch.from_numpy(synth.make_weights(rng, qt, n, kk)).cuda()

    x = torch.from_numpy(rng.standard_normal((m, k)).astype(np.float32)).to(dt).cuda()
    bias = torch.from_numpy(rng.standard_normal(96).astype(np.float32)).to(dt).cuda()
    for qt in (D.Q8_0, D.Q4_K, D.IQ4_XS):
        w = packed(qt, 96, k)
        _both(monkeypatch, lambda: D.fused_mul_mat_gguf(x, w, qt, bias=bias))
    # three shards of a merged layer: the first two are one matrix to the compiled call
    parts = [packed(D.Q4_K, 48, k), packed(D.Q4_K, 16, k), packed(D.Q6_K, 32, k)]
    w = torch.zeros(96, max(p.shape[1] for p in parts), dtype=torch.uint8, device="cuda")
    at, row = {}, 0
    for i, p in zip("qkv", parts):
        w[row:row + p.shape[0], :p.shape[1]] = p
        at[i] = (row, row + p.shape[0], p.shape[1])
        row += p.shape[0]
    types = {"q": D.Q4_K, "k": D.Q4_K, "v": D.Q6_K}
    _both(monkeypatch, lambda: D.apply_linear(x, w, D.Q4_K, shard_ids=("q", "k", "v"), shard_offset_map=at, shard_weight_types=types, bias=bias))
    w1 = packed(D.Q4_0, e * 2 * inner, k).reshape(e, 2 * inner, -1)
    w2 = packed(D.Q4_0, e * k, inner).reshape(e, k, -1)
    tw, ids = torch.topk(torch.softmax(torch.from_numpy(rng.standard_normal((m, e)).astype(np.float32)).cuda(), 1), top_k)
    _both(monkeypatch, lambda: D.fused_moe_gguf(x, w1, w2, tw, ids.to(torch.int32), D.Q4_0, D.Q4_0, "silu"))
    table = packed(D.Q6_K, 64, k)
    rows = torch.from_numpy(rng.integers(0, 64, size=(m, 2))).cuda()
    _both(monkeypatch, lambda: D.apply_gguf_embedding(rows, table, D.Q6_K, k, dt))


def test_workspace_is_that_of_the_engine_that_runs():
    from vllm_gguf_plugin_prism_amd import _lib, ops
    L = _lib.lib()

    def layer(qt, n, k, m):
        qk, size = ops.quant_sizes(qt)
        return L.gguf_mmq_layer_workspace_bytes(qt, n, k, m, k // qk * size)

    n, k, m = 4096, 14336, 2048
    int8 = L.gguf_mmq_workspace_bytes_engine(m, n, k, ops.MMQ_ENGINES["int8"])
    for qt in (D.Q8_0, D.Q4_0, D.Q3_K):                       # formats whose products stay on the int8 unit
        assert layer(qt, n, k, m) == int8
    assert layer(D.Q4_K, n, k, 64) == L.gguf_mmq_workspace_bytes_engine(64, n, k, ops.MMQ_ENGINES["int8"])
    # one form of the rows (halves, block scales, block sums) and at most two partial tiles per CU, not the int8 rows too
    assert m * 2 * k <= layer(D.Q4_K, n, k, m) <= m * (2 * (k + 640) + k // 8 + k // 16) + 256 * 2 * 256 * 128 * 4
