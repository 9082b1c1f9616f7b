"""The streaming tile kernel (csrc/tile_stream_core.h) at the sizes where its panels, chunks of K, column groups and blocks
of slots begin and end, against the CPU oracle."""
import numpy as np
import pytest
import torch

from oracle import gguf_oracle as o

pytestmark = pytest.mark.gpu

SHORT, DEEP = (o.Q4_0, o.Q8_0), (o.Q4_K, o.Q5_K, o.Q6_K)


# (dealt to the waves of a workgroup, all but one) one and two tiles of rows, full and with a row over; a last column group of one column; rows of X shorter than a panel,
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
                                                      (o.Q5_K, 24, 6, 4096, 256), (o.Q6_K, 24, 6, 4096, 768), (o.Q4_0, 60, 40, 736, 1056),
                                                      (o.Q8_0, 90, 44, 544, 2080), (o.Q4_K, 60, 40, 2304, 1024), (o.Q6_K, 40, 36, 1280, 1280), (o.Q5_K, 12, 6, 768, 512)])
def test_moe_layer_edges(qtype, tokens, e, hid, inner):
    check_layer(qtype, tokens, e, hid, inner)


def check_layer(qtype, tokens, e, hid, inner, routing=None):
    from vllm_gguf_plugin_prism_amd import ops
    rng = np.random.default_rng(hid + inner)
    top_k = 2
    w13 = np.stack([o.make_weights(rng, qtype, 2 * inner, hid) for _ in range(e)])
    w2 = np.stack([o.make_weights(rng, qtype, hid, inner) for _ in range(e)])
    ids = np.stack([rng.permutation(e)[:top_k] for _ in range(tokens)]).astype(np.int32) if routing is None else routing.copy()
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


# sizes that the cost rule sends here from the other kernels; all but the widest have their panels dealt to the waves of a workgroup (what is not:
# test_gpu_few_rows.py, test_kernels_of_what_is_not_dealt): more column groups than a round of workgroups holds and a last one in part, one and
# two tiles of rows, fewer rows than half a tile
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


# Layers of which both products deal K of their last blocks to two waves each: behind full rounds and from the first block on, an even and an odd
# number of panels, one of them in part, one panel per wave, inner sizes that end inside a workgroup's features.  Every expert is the same and
# so is every token: so are the results, bit for bit, whichever block a pair is in.
LAST_ROUND = [(o.Q4_0, 62, 4, 2016, 2048), (o.Q4_0, 42, 30, 1056, 1056), (o.Q4_K, 43, 6, 2304, 2048), (o.Q5_K, 34, 34, 2048, 512)]


def many_blocks(tokens, e):
    """Two experts per token so that as many blocks of 16 slots as possible hold pairs: one pair of every expert, then 16 more at a time."""
    count, left = np.ones(e, np.int64), 2 * tokens - e
    for i in range(left // 16 + 1):
        count[i % e] += min(16, left - 16 * i)
    return np.repeat(np.arange(e), count).reshape(tokens, 2).astype(np.int32)


def last_blocks(qtype, tokens, e, hid, inner, ids):
    """How many blocks with pairs have K dealt to two waves, in either product."""
    from vllm_gguf_plugin_prism_amd import _lib
    live = int(((np.bincount(ids[ids < e], minlength=e) + 15) // 16).sum())
    start = [_lib.lib().gguf_moe_mmq_layer_finer(qtype, qtype, hid, inner, hid, 2, tokens, e, product) for product in (1, 2)]
    return [live - at if at >= 0 else 0 for at in start]


@pytest.mark.parametrize("qtype,tokens,e,hid,inner", LAST_ROUND)
def test_moe_rows_do_not_depend_on_their_block(qtype, tokens, e, hid, inner):
    from vllm_gguf_plugin_prism_amd import ops
    rng = np.random.default_rng(hid)
    ids = many_blocks(tokens, e)
    assert min(last_blocks(qtype, tokens, e, hid, inner, ids)) > 0
    w13, w2 = (torch.from_numpy(o.make_weights(rng, qtype, *shape)).cuda().repeat(e, 1, 1) for shape in ((2 * inner, hid), (hid, inner)))
    x = torch.from_numpy(rng.standard_normal(hid).astype(np.float32)).cuda()[None]
    x = (x * (4.0 / ops.ggml_mul_mat_a8(w13[0], x, qtype, 2 * inner).abs().max())).repeat(tokens, 1)
    got = ops.moe_mmq_layer(x, w13, w2, torch.full((tokens, 2), 0.5, device="cuda"), torch.from_numpy(ids).cuda(), qtype, qtype, "silu")
    assert bool(got.isfinite().all()) and torch.equal(got, got[:1].repeat(tokens, 1))


@pytest.mark.parametrize("qtype,tokens,e,hid,inner", LAST_ROUND)
def test_moe_layer_last_round(qtype, tokens, e, hid, inner):
    ids = many_blocks(tokens, e)
    ids[3, 1] = e + 2
    assert min(last_blocks(qtype, tokens, e, hid, inner, ids)) > 0
    check_layer(qtype, tokens, e, hid, inner, ids)
