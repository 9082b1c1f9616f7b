"""What reaches the codebook formats' GEMM (csrc/dense_core.h) and what does not: ``fused_mul_mat_gguf`` takes every call that
a dense copy of the weights and ``x @ dense.T`` (then ``add_`` of the bias, ``copy_`` to the result) takes, with their
result, and refuses what they refuse, whether or not the number of rows is one that the GEMM serves."""
import numpy as np
import pytest
import torch

from vllm_gguf_plugin_prism_amd import dispatch as D
from vllm_gguf_plugin_prism_amd import ops, synth

pytestmark = pytest.mark.gpu
QT, N, K, M = D.IQ4_XS, 512, 512, 40         # (40 rows: the GEMM serves the plain call)


def _weights(pad=0):
    packed = torch.from_numpy(synth.make_weights(np.random.default_rng(1), QT, N, K)).cuda()
    w = torch.zeros(N, packed.shape[1] + pad, dtype=torch.uint8, device="cuda")
    w[:, :packed.shape[1]] = packed
    return w, packed


def _x(*shape, dtype=torch.float16, seed=2):
    return torch.from_numpy(np.random.default_rng(seed).standard_normal(shape).astype(np.float32)).to(dtype).cuda()


def _dense(packed, dtype=torch.float16):
    return ops.ggml_dequantize(packed, QT, N, K, dtype)


def _close(got, want, rel=1e-3):              # two roundings to 16 bits and a sum in another order
    assert got.shape == want.shape and got.dtype == want.dtype
    assert ((got.double() - want.double()).norm() / want.double().norm()).item() <= rel


def test_the_plain_call_is_served():
    w, _ = _weights()
    assert ops.dense_linear(w, _x(M, K), QT, N) is not None


@pytest.mark.parametrize("shape", [(M, 3, K), (M, 1, K)])
def test_activations_of_three_dimensions(shape):
    w, packed = _weights()
    x = _x(*shape)
    _close(D.fused_mul_mat_gguf(x, w, QT), x @ _dense(packed).T)


@pytest.mark.parametrize("bias", ["fp32", "one", "row"])
def test_a_bias_that_add_takes(bias):
    w, packed = _weights()
    x = _x(M, K)
    b = {"fp32": _x(N, dtype=torch.float32), "one": _x(1), "row": _x(1, N)}[bias]
    _close(D.fused_mul_mat_gguf(x, w, QT, bias=b), (x @ _dense(packed).T).add_(b))


def test_a_result_that_copy_takes():
    w, packed = _weights()
    x = _x(M, K)
    want = x @ _dense(packed).T
    for out in (torch.empty(M, N, device="cuda"), torch.empty(N, M, dtype=x.dtype, device="cuda").T, torch.empty(2, M, N, dtype=x.dtype, device="cuda")):
        got = D.fused_mul_mat_gguf(x, w, QT, out=out)
        assert got is out
        _close(got, want.to(out.dtype).expand(out.shape))


def test_a_result_over_the_activations():      # (N == K)
    w, packed = _weights()
    same = _x(M, K)
    want = same @ _dense(packed).T
    _close(D.fused_mul_mat_gguf(same, w, QT, out=same), want)


def test_a_result_whose_rows_overlap_is_refused():
    w, _ = _weights()
    with pytest.raises(RuntimeError):
        D.fused_mul_mat_gguf(_x(M, K), w, QT, out=torch.empty(1, N, dtype=torch.float16, device="cuda").expand(M, N))


def test_weights_of_another_width_are_refused():
    block = ops.quant_sizes(QT)[1]
    wide, _ = _weights(pad=block)
    for dtype in (torch.float16, torch.float32):   # (the GEMM takes no 32-bit activations)
        with pytest.raises(RuntimeError):
            D.fused_mul_mat_gguf(_x(M, K, dtype=dtype), wide, QT)
    at, x = {"gate": (0, N, wide.shape[1]), "up": (0, N, wide.shape[1])}, _x(M, K)
    with pytest.raises(RuntimeError):
        D.apply_linear(x, wide, QT, shard_ids=("gate", "up"), shard_offset_map=at, shard_weight_types={"gate": QT, "up": D.IQ2_S})


def test_bytes_behind_the_last_block_are_no_weights():
    padded, packed = _weights(pad=6)
    for dtype in (torch.float16, torch.float32):
        x = _x(M, K, dtype=dtype)
        _close(D.fused_mul_mat_gguf(x, padded, QT), x @ _dense(packed, dtype).T)


def test_packed_weights_of_another_integer_type():
    w, packed = _weights()
    x = _x(M, K)
    _close(D.fused_mul_mat_gguf(x, w.view(torch.int8), QT), x @ _dense(packed).T)


# ---- what torch does in the product of a dense copy beyond multiplying


def test_gradients_reach_the_activations_and_the_bias():
    w, packed = _weights()
    for dtype in (torch.float16, torch.float32):
        got, want = [], []
        for kept, product in ((got, lambda x, b: D.fused_mul_mat_gguf(x, w, QT, bias=b)), (want, lambda x, b: (x @ _dense(packed, dtype).T).add_(b))):
            x, b = _x(M, K, dtype=dtype).requires_grad_(), _x(N, dtype=dtype, seed=3).requires_grad_()
            y = product(x, b)
            assert y.requires_grad
            y.backward(_x(M, N, dtype=dtype, seed=5))
            kept += [y.detach(), x.grad, b.grad]
        for g, r in zip(got, want):
            _close(g, r)
    with torch.no_grad():
        assert not D.fused_mul_mat_gguf(_x(M, K).requires_grad_(), w, QT).requires_grad


def test_gradients_through_a_merged_layer():
    w, packed = _weights()
    at, types = {"gate": (0, 256, w.shape[1]), "up": (256, N, ops.quant_sizes(D.IQ4_NL)[1] * K // 32)}, {"gate": QT, "up": D.IQ4_NL}
    wide = torch.zeros(N, max(v[2] for v in at.values()), dtype=torch.uint8, device="cuda")
    wide[:256, :w.shape[1]] = w[:256]
    nl = torch.from_numpy(synth.make_weights(np.random.default_rng(4), D.IQ4_NL, 256, K)).cuda()
    wide[256:, :nl.shape[1]] = nl
    dense = torch.cat([_dense(packed)[:256], ops.ggml_dequantize(nl, D.IQ4_NL, 256, K, torch.float16)])
    x = _x(M, K).requires_grad_()
    y = D.apply_linear(x, wide, QT, shard_ids=("gate", "up"), shard_offset_map=at, shard_weight_types=types)
    _close(y.detach(), x.detach() @ dense.T)
    y.backward(torch.ones_like(y))
    _close(x.grad, torch.ones_like(y) @ dense)


def test_tangents_are_carried_along():
    import torch.autograd.forward_ad as fwd
    w, packed = _weights()
    with fwd.dual_level():
        y = D.fused_mul_mat_gguf(fwd.make_dual(_x(M, K), _x(M, K, seed=4)), w, QT)
        _close(fwd.unpack_dual(y).tangent, _x(M, K, seed=4) @ _dense(packed).T)


def test_vmap():
    w, packed = _weights()
    x = _x(3, M, K)
    _close(torch.func.vmap(lambda v: D.fused_mul_mat_gguf(v, w, QT))(x), x @ _dense(packed).T)


def test_autocast():
    w, packed = _weights()
    x = _x(M, K)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        got = D.fused_mul_mat_gguf(x, w, QT)
        _close(got, x @ _dense(packed).T, 8e-3)
    assert got.dtype == torch.bfloat16


def test_subclasses_and_modes_see_the_product():
    class Marked(torch.Tensor):
        pass

    from torch.utils.flop_counter import FlopCounterMode

    w, _ = _weights()
    assert type(D.fused_mul_mat_gguf(_x(M, K).as_subclass(Marked), w, QT)) is Marked
    with FlopCounterMode(display=False) as counter:
        D.fused_mul_mat_gguf(_x(M, K), w, QT)
    assert counter.get_total_flops() == 2 * M * N * K


def test_a_result_that_a_graph_has_saved():
    w, _ = _weights()
    out, p = _x(M, N), torch.ones(M, N, dtype=torch.float16, device="cuda", requires_grad=True)
    y = p * out
    D.fused_mul_mat_gguf(_x(M, K), w, QT, out=out)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        y.backward(torch.ones_like(y))
