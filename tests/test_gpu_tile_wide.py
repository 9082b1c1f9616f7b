"""The wide tile kernel (csrc/tile_wide_core.h) at the edges of its tiles of rows, columns and parts of K, and in MoE layers
whose experts see more than a few pairs each, against the CPU oracle."""
import numpy as np
import pytest
import torch

from oracle import gguf_oracle as o

pytestmark = pytest.mark.gpu

DENSE = (o.Q4_0, o.Q4_K, o.Q5_K, o.Q6_K, o.Q2_K, o.Q3_K, o.Q4_1, o.Q5_1)
ONES = (o.Q4_1, o.Q5_1)


# one row over a tile of 32 and of 64; a last column tile of one, four, some columns; one panel, K in one part and in
# several, a part that is longer than another; more tiles than a round of workgroups; rows of W a pitch apart that moves
# them through the positions inside 16 bytes (whole 16 bytes where only those are taken)
@pytest.mark.parametrize("qtype", DENSE)
@pytest.mark.parametrize("m,n,k,pad", [(513, 1025, 256, 0), (577, 1300, 768, 2), (33, 4101, 4096, 0), (513, 2052, 512, 6), (577, 256, 8192, 0),
                                       (40, 8196, 2048, 0), (97, 25604, 256, 0)])
def test_dense_edges(qtype, m, n, k, pad):
    check_dense(qtype, m, n, k, 8 * pad if qtype in ONES else pad)


# the last panel has one block, four, seven; K in one part and in several; more rows than other types are taken with
@pytest.mark.parametrize("qtype,m,n,k", [(o.Q4_1, 545, 640, 2176), (o.Q4_1, 577, 1300, 896), (o.Q5_1, 513, 2052, 1600), (o.Q5_1, 577, 256, 2496),
                                         (o.Q4_1, 521, 300, 384), (o.Q2_K, 2100, 130, 256), (o.Q5_1, 2100, 130, 320)])
def test_last_panels(qtype, m, n, k):
    check_dense(qtype, m, n, k, 0)


# a workspace for half of the rows: two passes (the oracle on rows of both, of the second's last tile)
def test_two_passes():
    from vllm_gguf_plugin_prism_amd import _lib
    m, n, k = 2041, 2052, 3072
    assert _lib.lib().gguf_mmq_layer_workspace_bytes(o.Q2_K, n, k, m, k // 256 * 84) < k // 128 * m * 272
    check_dense(o.Q2_K, m, n, k, 0, np.r_[:3, 1020:1030, m - 30:m])


# the half-precision unit where it is still the fastest: a row and a column over a tile, tiles cut into runs; whole rounds and a
# shared rest (the oracle on rows of several tiles)
@pytest.mark.parametrize("qtype", (o.Q4_K, o.Q5_K, o.Q6_K))
@pytest.mark.parametrize("m,n,k,pad", [(511, 2177, 8192, 2), (700, 2176, 5120, 0)])
def test_half_precision_unit_behind_them(qtype, m, n, k, pad):
    check_dense(qtype, m, n, k, pad, np.r_[:3, 250:260, m - 30:m], 2)


def check_dense(qtype, m, n, k, pad, rows=np.s_[:], unit=None):
    from vllm_gguf_plugin_prism_amd import ops
    rng = np.random.default_rng(n + m)
    w = o.make_weights(rng, qtype, n, k)
    wd = torch.zeros(n, w.shape[1] + pad, dtype=torch.uint8, device="cuda")[:, :w.shape[1]]
    wd.copy_(torch.from_numpy(w))
    assert ops._mmq_unit(qtype, n, k, m, wd.stride(0)) & 4 if unit is None else ops._mmq_unit(qtype, n, k, m, wd.stride(0)) == unit
    x = rng.standard_normal((m, k)).astype(np.float32) + 0.3
    bias = rng.standard_normal(n).astype(np.float32)
    y = ops.ggml_mul_mat_a8(wd, torch.from_numpy(x).cuda(), qtype, n, bias=torch.from_numpy(bias).cuda())
    assert o.rel_l2(y.cpu().numpy()[rows], o.mul_mat_a8(w, x[rows], qtype, n, "mmq") + bias) <= 1e-5


# the largest operands and sums, and scales that are subnormal halves (an offset that is rounded away would be all of it)
@pytest.mark.parametrize("qtype", DENSE)
def test_largest_sums_and_smallest_scales(qtype):
    from vllm_gguf_plugin_prism_amd import ops
    rng = np.random.default_rng(qtype)
    n, k, m = 384, 512, 520
    block, size = o.QUANT_SIZES[qtype]
    w = o.make_weights(rng, qtype, n, k).reshape(n, k // block, size)
    if qtype == o.Q6_K:
        w[:, :, :192], w[:, :, 192:208] = 0, 0x80          # codes -32, scales -128
        w[::2, :, 208:210] = np.frombuffer(np.float16(3e-6).tobytes(), np.uint8)
    elif qtype in (o.Q2_K, o.Q3_K):
        at = size - (4 if qtype == o.Q2_K else 2)          # (scales 31 for Q3_K, codes -4 where its third bits are clear)
        w[:, :, :at] = 0xFF
        if qtype == o.Q3_K:
            w[1::3, :, :96] = 0
        w[::2, :, at : at + 2] = np.frombuffer(np.float16(3e-6).tobytes(), np.uint8)
    else:
        w[:, :, 4 if qtype != o.Q4_0 else 2:] = 0xFF
        w[::2, :, :2] = np.frombuffer(np.float16(3e-6).tobytes(), np.uint8)
    w = w.reshape(n, -1)
    x = rng.choice([-1.0, 1.0], size=(m, k)).astype(np.float32) * 3.0
    x[: m // 2] = np.abs(x[: m // 2])
    y = ops.ggml_mul_mat_a8(torch.from_numpy(w).cuda(), torch.from_numpy(x).cuda(), qtype, n).cpu().numpy()
    want = o.mul_mat_a8(w, x, qtype, n, "mmq")
    for part in (np.s_[::2], np.s_[1::2]):
        assert o.rel_l2(y[:, part], want[:, part]) <= 1e-5


# blocks of slots full and in part, an expert without pairs, a pair whose expert does not exist; the second product's K in
# one part and in two; a hidden size that ends inside a column tile
@pytest.mark.parametrize("qtype,qtype2,tokens,e,hid,inner", [
    (o.Q4_0, o.Q4_0, 200, 5, 256, 1024), (o.Q8_0, o.Q4_0, 150, 4, 512, 1792), (o.Q4_K, o.Q6_K, 200, 5, 256, 1024), (o.Q5_K, o.Q5_K, 150, 4, 768, 1536),
    (o.Q6_K, o.Q8_0, 150, 4, 512, 1792), (o.Q4_K, o.Q4_K, 130, 4, 512, 2048)])
def test_moe_layer(qtype, qtype2, tokens, e, hid, inner):
    from vllm_gguf_plugin_prism_amd import _lib, ops
    rng = np.random.default_rng(hid + inner)
    top_k = 2
    assert _lib.lib().gguf_moe_mmq_layer_wide(qtype, qtype2, hid, inner, hid, top_k, tokens, e) == 1
    w13 = np.stack([o.make_weights(rng, qtype, 2 * inner, hid) for _ in range(e)])
    w2 = np.stack([o.make_weights(rng, qtype2, hid, inner) for _ in range(e)])
    ids = np.stack([rng.permutation(e - 1)[:top_k] for _ in range(tokens)]).astype(np.int32)
    ids[3, 1] = e + 2
    wts = rng.random((tokens, top_k)).astype(np.float32)
    x = rng.standard_normal((tokens, hid)).astype(np.float32)
    s, eids, post = o.moe_align_block_size(ids, 32, e)
    h = o.moe_a8(x, w13, s, eids, post, qtype, 2 * inner, top_k, tokens, 32)
    x *= 4.0 / np.abs(h).max()
    h = o.moe_a8(x, w13, s, eids, post, qtype, 2 * inner, top_k, tokens, 32)
    y = o.moe_a8(o.silu_and_mul(h), w2, s, eids, post, qtype2, hid, 1, tokens * top_k, 32)
    want = (y.reshape(tokens, top_k, hid) * wts[:, :, None]).sum(1)
    cuda = [torch.from_numpy(a).cuda() for a in (x, w13, w2, wts, ids)]
    got = ops.moe_mmq_layer(*cuda, qtype, qtype2, "silu")
    # (a quant of h may move by a step where the activation's last bit differs)
    assert o.rel_l2(got.cpu().numpy(), want) <= 1e-3
