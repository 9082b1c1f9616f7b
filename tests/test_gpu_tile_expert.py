"""The expert tile kernel (csrc/tile_expert_core.h): blocks of 32 slots with one pair, sixteen, seventeen and all, against the CPU oracle."""
import numpy as np
import pytest
import torch

from oracle import gguf_oracle as o
from test_gpu_tile_wide import layer

pytestmark = pytest.mark.gpu


# either kind of record behind either kernel; a column tile of one feature's run, of some; K in one part and in four; pairs whose expert
# does not exist; an infinite block scale in a block of 17 pairs and in one of one: that row holds a number, an infinity or neither
# where the other kernels' does, its neighbours are numbers
@pytest.mark.parametrize("qtype,qtype2,hid,inner,n_out", [
    (o.Q4_0, o.Q4_0, 256, 768, 256), (o.Q8_0, o.Q8_0, 512, 6144, 129), (o.Q4_K, o.Q4_K, 256, 1536, 130), (o.Q5_K, o.Q5_K, 768, 768, 384),
    (o.Q4_K, o.Q6_K, 256, 768, 256), (o.Q6_K, o.Q5_K, 512, 1536, 131), (o.Q6_K, o.Q6_K, 256, 6144, 252)])
@pytest.mark.parametrize("huge", (False, True))
def test_blocks_in_part(qtype, qtype2, hid, inner, n_out, huge):
    from vllm_gguf_plugin_prism_amd import _lib, ops
    rng = np.random.default_rng(hid + inner + n_out)
    pairs_of = (1, 16, 17, 32, 33, 0, 209)                  # by expert; a block with 1, 16, 17, 32, 1 and 17 pairs
    e, tokens = len(pairs_of), sum(pairs_of) + 1
    w13 = np.stack([o.make_weights(rng, qtype, 2 * inner, hid) for _ in range(e)])
    w2 = np.stack([o.make_weights(rng, qtype2, n_out, inner) for _ in range(e)])
    ids = np.append(np.repeat(np.arange(e), pairs_of), e + 3).astype(np.int32)
    order = rng.permutation(tokens)
    ids = ids[order][:, None].copy()
    assert _lib.lib().gguf_moe_mmq_layer_wide(qtype, qtype2, hid, inner, n_out, 1, tokens, e) == 1
    x = rng.standard_normal((tokens, hid)).astype(np.float32)
    wts = rng.random((tokens, 1)).astype(np.float32)
    s, eids, post = o.moe_align_block_size(ids, 32, e)
    h = o.moe_a8(x, w13, s, eids, post, qtype, 2 * inner, 1, tokens, 32)
    x *= 4.0 / np.abs(h).max()
    rows = [int(np.flatnonzero(ids[:, 0] == j)[0]) for j in (0, 2)] if huge else []
    for r in rows:
        x[r, 40] = 1e8                                      # (its block's scale, 1e8 / 127, is infinite as a half)
    cuda = [torch.from_numpy(a).cuda() for a in (x, w13, w2, wts, ids)]
    got = ops.moe_mmq_layer(*cuda, qtype, qtype2, "silu").cpu().numpy()
    with np.errstate(all="ignore"):
        h = o.moe_a8(x, w13, s, eids, post, qtype, 2 * inner, 1, tokens, 32)
        y = o.moe_a8(o.silu_and_mul(h), w2, s, eids, post, qtype2, n_out, 1, tokens, 32)
        want = y * wts
    rest = np.setdiff1d(np.arange(tokens), rows)
    # (a quant of h may move by a step where the activation's last bit differs)
    assert np.isfinite(got[rest]).all() and o.rel_l2(got[rest], want[rest]) <= 1e-3
    if rows and qtype != o.Q6_K:                            # (the other route: a workspace off 16 bytes; the wide tiles of Q6_K differ from it there)
        other = layer("gguf_moe_mmq_layer", *cuda, qtype, qtype2, 8).cpu().numpy()
        for r in rows:
            assert (np.isnan(got[r]) == np.isnan(other[r])).all() and (np.isinf(got[r]) == np.isinf(other[r])).all()


# rows that hold an activation that is no number, some in every block: they are not walked again, as a row whose block scale is infinite is (that is 1.7 times the
# layer's time); the rows beside them keep their bits
@pytest.mark.parametrize("qtype", (o.Q4_K, o.Q4_0))
def test_rows_without_numbers_take_one_walk(qtype):
    from vllm_gguf_plugin_prism_amd import _lib
    rng = np.random.default_rng(qtype)
    tokens, e, hid, inner = 600, 8, 2048, 1024
    assert _lib.lib().gguf_moe_mmq_layer_wide(qtype, qtype, hid, inner, hid, 1, tokens, e) == 1
    w13 = np.stack([o.make_weights(rng, qtype, 2 * inner, hid) for _ in range(e)])
    w2 = np.stack([o.make_weights(rng, qtype, hid, inner) for _ in range(e)])
    ids, wts = rng.permutation(np.arange(tokens) % e).astype(np.int32)[:, None].copy(), rng.random((tokens, 1)).astype(np.float32)
    x = torch.from_numpy(0.01 * rng.standard_normal((tokens, hid)).astype(np.float32)).cuda()
    rest = [torch.from_numpy(a).cuda() for a in (w13, w2, wts, ids)]
    none = torch.zeros(tokens, dtype=torch.bool, device="cuda")
    none[::6] = True
    with_none = x.clone()
    with_none[none, 1000] = float("nan")
    want, us = layer("gguf_moe_mmq_layer", x, *rest, qtype, qtype), {}
    got = layer("gguf_moe_mmq_layer", with_none, *rest, qtype, qtype)
    assert torch.equal(got[~none], want[~none]) and bool(got[none].isnan().any(1).all()) and bool(want.isfinite().all())
    L, out = _lib.lib(), torch.empty_like(x)
    nbytes = L.gguf_moe_mmq_layer_workspace_bytes(qtype, qtype, tokens, 1, hid, inner, hid, e, 0)
    ws = torch.empty(nbytes, dtype=torch.uint8, device="cuda")
    for rows in (x, with_none) * 10:
        begin, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
        begin.record()
        for _ in range(10):
            assert L.gguf_moe_mmq_layer(rows.data_ptr(), 0, rest[0].data_ptr(), qtype, rest[1].data_ptr(), qtype, rest[3].data_ptr(), rest[2].data_ptr(), ws.data_ptr(), nbytes,
                                        out.data_ptr(), hid, inner, hid, 1, tokens, 1, e, torch.cuda.current_stream().cuda_stream) == 0
        end.record()
        end.synchronize()
        us[rows is x] = min(us.get(rows is x, 1e9), begin.elapsed_time(end) * 100.0)
    assert us[False] < 1.25 * us[True], us


# two experts with the same weights, the rows of one, three to sixteen of a block, among those of the other, which fill theirs: the same bits, tiles of 16 x 16 or of
# 32 x 32 (activations of one sign too, whose offsets are as large as the products)
@pytest.mark.parametrize("qtype,qtype2", [(o.Q4_0, o.Q4_0), (o.Q8_0, o.Q8_0), (o.Q4_K, o.Q4_K), (o.Q5_K, o.Q5_K), (o.Q6_K, o.Q6_K)])
@pytest.mark.parametrize("few", (3, 16))
@pytest.mark.parametrize("one_sign", (False, True))
def test_a_pair_has_the_bits_it_has_in_a_full_block(qtype, qtype2, few, one_sign):
    from vllm_gguf_plugin_prism_amd import _lib
    rng = np.random.default_rng(qtype + few)
    e, hid, inner, full = 3, 768, 1024, 32
    counts = (few, full, 150)
    tokens = sum(counts)
    assert _lib.lib().gguf_moe_mmq_layer_wide(qtype, qtype2, hid, inner, hid, 1, tokens, e) == 1
    w13 = np.stack([o.make_weights(rng, qtype, 2 * inner, hid)] * 2 + [o.make_weights(rng, qtype, 2 * inner, hid)])
    w2 = np.stack([o.make_weights(rng, qtype2, hid, inner)] * 2 + [o.make_weights(rng, qtype2, hid, inner)])
    x = 0.05 * rng.standard_normal((tokens, hid)).astype(np.float32)
    x = 0.02 * np.abs(x) if one_sign else x                 # (so that sums of h fit in a half)
    x[few:2 * few] = x[:few]
    ids = np.repeat(np.arange(e), counts).astype(np.int32)[:, None].copy()
    cuda = [torch.from_numpy(a).cuda() for a in (x, w13, w2, np.ones((tokens, 1), np.float32), ids)]
    got = layer("gguf_moe_mmq_layer", *cuda, qtype, qtype2)
    assert bool(got.isfinite().all()) and torch.equal(got[:few], got[few:2 * few])
