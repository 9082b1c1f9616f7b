"""The streaming tile kernel (csrc/tile_stream_core.h) at the sizes where its panels, chunks of K, column groups and blocks
of slots begin and end, against the CPU oracle."""
import numpy as np
import pytest
import torch

from oracle import gguf_oracle as o

pytestmark = pytest.mark.gpu

SHORT, DEEP = (o.Q4_0, o.Q8_0), (o.Q4_K, o.Q5_K, o.Q6_K)


# one and two tiles of rows, full and with a row over; a last column group of one column; rows of X shorter than a panel,
# ending inside one, in one chunk, in two, in more than a chunk's double buffer; rows of W a pitch apart that moves them
# through all positions inside 16 bytes
@pytest.mark.parametrize("qtype,m,n,k,pad", [(q, *s) for q in SHORT for s in (
    (9, 40, 32, 0), (16, 513, 736, 0), (17, 48, 1312, 2), (32, 2049, 288, 0), (12, 72, 5152, 0), (20, 2064, 4640, 6), (7, 2100, 5120, 0))] + [
    (q, *s) for q in DEEP for s in ((9, 33, 256, 0), (17, 513, 1280, 4), (16, 100, 4096, 2), (32, 4112, 8192, 0))])
def test_dense_edges(qtype, m, n, k, pad):
    from vllm_gguf_plugin_prism_amd import ops
    rng = np.random.default_rng(n + m)
    w = o.make_weights(rng, qtype, n, k)
    wd = torch.zeros(n, w.shape[1] + pad, dtype=torch.uint8, device="cuda")[:, :w.shape[1]]
    wd.copy_(torch.from_numpy(w))
    x = rng.standard_normal((m, k)).astype(np.float32)
    bias = rng.standard_normal(n).astype(np.float32)
    y = ops.ggml_mul_mat_a8(wd, torch.from_numpy(x).cuda(), qtype, n, bias=torch.from_numpy(bias).cuda())
    assert o.rel_l2(y.cpu().numpy(), o.mul_mat_a8(w, x, qtype, n, "mmq") + bias) <= 1e-5


# a few pairs per expert and enough experts that a wave walks two (or four) column groups; inner sizes that end inside a
# workgroup's features; the longest K of the gated product; a pair whose expert does not exist
@pytest.mark.parametrize("qtype,tokens,e,hid,inner", [(o.Q4_0, 60, 40, 288, 1056), (o.Q8_0, 24, 6, 4096, 800), (o.Q4_K, 60, 40, 256, 1280),
                                                      (o.Q5_K, 24, 6, 4096, 256), (o.Q6_K, 24, 6, 4096, 768)])
def test_moe_layer_edges(qtype, tokens, e, hid, inner):
    from vllm_gguf_plugin_prism_amd import ops
    rng = np.random.default_rng(hid + inner)
    top_k = 2
    w13 = np.stack([o.make_weights(rng, qtype, 2 * inner, hid) for _ in range(e)])
    w2 = np.stack([o.make_weights(rng, qtype, hid, inner) for _ in range(e)])
    ids = np.stack([rng.permutation(e)[:top_k] for _ in range(tokens)]).astype(np.int32)
    ids[3, 1] = e + 2
    wts = rng.random((tokens, top_k)).astype(np.float32)
    x = rng.standard_normal((tokens, hid)).astype(np.float32)
    s, eids, post = o.moe_align_block_size(ids, 16, e)
    h = o.moe_a8(x, w13, s, eids, post, qtype, 2 * inner, top_k, tokens, 16)
    x *= 4.0 / np.abs(h).max()
    h = o.moe_a8(x, w13, s, eids, post, qtype, 2 * inner, top_k, tokens, 16)
    y = o.moe_a8(o.silu_and_mul(h), w2, s, eids, post, qtype, hid, 1, tokens * top_k, 16)
    want = (y.reshape(tokens, top_k, hid) * wts[:, :, None]).sum(1)
    cuda = [torch.from_numpy(a).cuda() for a in (x, w13, w2, wts, ids)]
    got = ops.moe_mmq_layer(*cuda, qtype, qtype, "silu")
    # (a quant of h may move by a step where the activation's last bit differs)
    assert o.rel_l2(got.cpu().numpy(), want) <= 1e-3


# sizes that the cost rule sends here: more column groups than a round of workgroups holds and a last one in part, K in
# chunks, one and two tiles of rows, fewer rows than half a tile
@pytest.mark.parametrize("qtype,m,n,k", [(q, *s) for q in DEEP for s in ((5, 5200, 4352), (24, 5205, 4096), (8, 12300, 2304), (16, 28688, 512))] + [
    (o.Q4_0, 12, 2560, 4096), (o.Q8_0, 24, 2048, 8192)])
def test_dense_where_it_is_taken(qtype, m, n, k):
    from vllm_gguf_plugin_prism_amd import ops
    rng = np.random.default_rng(n + m)
    w = o.make_weights(rng, qtype, n, k)
    assert ops._mmq_route(qtype, n, k, m, w.shape[1]) == 1
    x = rng.standard_normal((m, k)).astype(np.float32)
    y = ops.ggml_mul_mat_a8(torch.from_numpy(w).cuda(), torch.from_numpy(x).cuda(), qtype, n)
    assert o.rel_l2(y.cpu().numpy(), o.mul_mat_a8(w, x, qtype, n, "mmq")) <= 1e-5


# layers whose last round of workgroups is cut finer: behind a full round in both products, an odd number of panels dealt to two waves,
# more blocks than expected, inner sizes that end inside a workgroup's features; all of a product in one round
@pytest.mark.parametrize("qtype,tokens,e,hid,inner", [(o.Q4_0, 60, 40, 736, 1056), (o.Q8_0, 90, 44, 544, 2080), (o.Q4_K, 60, 40, 2304, 1024), (o.Q6_K, 40, 36, 1280, 1280),
                                                      (o.Q5_K, 12, 6, 768, 512)])
def test_moe_layer_last_round(qtype, tokens, e, hid, inner):
    test_moe_layer_edges(qtype, tokens, e, hid, inner)
