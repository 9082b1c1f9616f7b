"""The wide tile kernel (csrc/tile_wide_core.h) at the edges of its tiles of rows, columns and parts of K, and in MoE layers
whose experts see more than a few pairs each, against the CPU oracle."""
import numpy as np
import pytest
import torch

from oracle import gguf_oracle as o

pytestmark = pytest.mark.gpu

DENSE = (o.Q4_0, o.Q4_K, o.Q5_K, o.Q6_K, o.Q2_K, o.Q3_K, o.Q4_1, o.Q5_1)
ONES = (o.Q4_1, o.Q5_1)
WALKED = (o.Q4_0, o.Q4_K, o.Q5_K, o.Q6_K, o.Q3_K)   # (the walking tiles take most of their sizes)


# one row over a tile of 32 and of 64; a last column tile of one, four, some columns; one panel, K in one part and in
# several, a part that is longer than another; more tiles than a round of workgroups; rows of W a pitch apart that moves
# them through the positions inside 16 bytes (whole 16 bytes where only those are taken)
@pytest.mark.parametrize("qtype,m,n,k,pad", [(q, *s) for q in DENSE if q not in WALKED for s in (
    (513, 1025, 256, 0), (577, 1300, 768, 2), (33, 4101, 4096, 0), (513, 2052, 512, 6), (577, 256, 8192, 0), (40, 8196, 2048, 0), (97, 25604, 256, 0))] + [
    (q, *s) for q in WALKED for s in ((783, 1145, 256, 0), (38, 760, 15872, 2), (581, 106, 9216, 6), (33, 16527, 2304, 0), (97, 25604, 256, 0))] + [
    (q, 513, 2052, 512, 6) for q in (o.Q4_0, o.Q4_K, o.Q6_K)])
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
@pytest.mark.parametrize("qtype,m,n,k,pad", [(q, *s) for q in (o.Q4_K, o.Q5_K) for s in ((2051, 513, 8192, 2), (2100, 2176, 5120, 0))] + [
    (o.Q6_K, 511, 2177, 8192, 2), (o.Q6_K, 700, 2176, 5120, 0)])
def test_half_precision_unit_behind_them(qtype, m, n, k, pad):
    check_dense(qtype, m, n, k, pad, np.r_[:3, 250:260, m - 30:m], 2)


def check_dense(qtype, m, n, k, pad, rows=np.s_[:], unit=4):
    from vllm_gguf_plugin_prism_amd import ops
    rng = np.random.default_rng(n + m)
    w = o.make_weights(rng, qtype, n, k)
    wd = torch.zeros(n, w.shape[1] + pad, dtype=torch.uint8, device="cuda")[:, :w.shape[1]]
    wd.copy_(torch.from_numpy(w))
    assert ops._mmq_route(qtype, n, k, m, wd.stride(0)) == unit and ops._linear_walk(qtype, n, k, m, wd.stride(0)) == (0, 0)
    x = rng.standard_normal((m, k)).astype(np.float32) + 0.3
    bias = rng.standard_normal(n).astype(np.float32)
    y = ops.ggml_mul_mat_a8(wd, torch.from_numpy(x).cuda(), qtype, n, bias=torch.from_numpy(bias).cuda())
    assert o.rel_l2(y.cpu().numpy()[rows], o.mul_mat_a8(w, x[rows], qtype, n, "mmq") + bias) <= 1e-5


# 16-bit results in columns of a wider tensor (from an odd one on: single stores): K in parts with a ragged N, in one part, two
# passes over the rows
@pytest.mark.parametrize("dt", (torch.float16, torch.bfloat16))
@pytest.mark.parametrize("qtype,m,n,k,column", [(q, *s) for q in (o.Q2_K, o.Q4_1, o.Q5_1) for s in ((33, 4101, 4096, 3), (577, 1300, 768, 4))] + [
    (q, *s) for q in (o.Q4_0, o.Q3_K) for s in ((34, 1010, 12288, 3), (783, 1145, 256, 4))] + [(o.Q2_K, 2041, 2052, 3072, 1)])
def test_16_bit_results(qtype, m, n, k, column, dt):
    from vllm_gguf_plugin_prism_amd import ops
    rng = np.random.default_rng(n + m)
    rows = np.r_[:33] if m < 2000 else np.r_[:3, 1020:1030, m - 30:m]
    w = o.make_weights(rng, qtype, n, k)
    assert ops._mmq_route(qtype, n, k, m, w.shape[1]) == 4 and ops._linear_walk(qtype, n, k, m, w.shape[1]) == (0, 0)
    x = torch.from_numpy(rng.standard_normal((m, k)).astype(np.float32)).to(dt)
    bias = torch.from_numpy(rng.standard_normal(n).astype(np.float32)).to(dt)
    wide = torch.full((m, column + n + 4), 7.0, dtype=dt, device="cuda")
    out = ops.ggml_mul_mat_a8(torch.from_numpy(w).cuda(), x.cuda(), qtype, n, out=wide[:, column:column + n], bias=bias.cuda())
    want = o.mul_mat_a8(w, x[rows].float().numpy(), qtype, n, "mmq") + bias.float().numpy()
    # two roundings to 16 bits (product, product plus bias), each half a unit in the last place of 11 or 8 bits
    assert o.rel_l2(out[rows].float().cpu().numpy(), want) <= {torch.float16: 2.0 ** -10, torch.bfloat16: 2.0 ** -7}[dt]
    assert bool((wide[:, :column] == 7).all()) and bool((wide[:, column + n:] == 7).all())


# the largest operands and sums, and scales that are subnormal halves (an offset that is rounded away would be all of it)
# (the last sizes: the walking tiles)
@pytest.mark.parametrize("qtype,m,n", [(q, 520, 384) for q in DENSE if q not in WALKED] + [(q, 33, 23472) for q in WALKED] + [(q, 520, 384) for q in WALKED])
def test_largest_sums_and_smallest_scales(qtype, m, n):
    from vllm_gguf_plugin_prism_amd import ops
    rng = np.random.default_rng(qtype)
    k = 512
    assert (ops._linear_walk(qtype, n, k, m, k // ops.quant_sizes(qtype)[0] * ops.quant_sizes(qtype)[1]) != (0, 0)) == (qtype in WALKED and m == 520)
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


def layer(entry, x, w13, w2, wts, ids, t13, t2, off=0, nbytes=None):
    """A layer's entry point of the C ABI with a workspace that begins `off` bytes behind a 16-byte boundary; nbytes: its size,
    else what the entry point asks for."""
    from vllm_gguf_plugin_prism_amd import _lib
    L = _lib.lib()
    (tokens, top_k), hid, inner, n_out, e = ids.shape, x.shape[1], w13.shape[1] // 2, w2.shape[1], w13.shape[0]
    code = {torch.float32: 0, torch.float16: 1, torch.bfloat16: 2}[x.dtype]
    types = (t13, t2) if entry == "gguf_moe_mmq_layer" else ()
    nbytes = nbytes or getattr(L, entry + "_workspace_bytes")(*types, tokens, top_k, hid, inner, n_out, e, code)
    ws = torch.full((nbytes + 32,), 0xFF, dtype=torch.uint8, device="cuda")
    out = torch.full((tokens, n_out), 7.0, dtype=x.dtype, device="cuda")
    assert ws.data_ptr() % 16 == 0
    rc = getattr(L, entry)(x.data_ptr(), code, w13.data_ptr(), t13, w2.data_ptr(), t2, ids.data_ptr(), wts.data_ptr(), ws.data_ptr() + off,
                           nbytes, out.data_ptr(), hid, inner, n_out, top_k, tokens, 1, e, torch.cuda.current_stream().cuda_stream)
    assert rc == 0 and (ws[nbytes + off:] == 0xFF).all() and (ws[:off] == 0xFF).all()
    return out


def layer_inputs(rng, t13, t2, tokens, e, hid, inner, dtype, n_out=None):
    w13 = np.stack([o.make_weights(rng, t13, 2 * inner, hid) for _ in range(e)])
    w2 = np.stack([o.make_weights(rng, t2, n_out or hid, inner) for _ in range(e)])
    ids = np.stack([rng.permutation(e)[:2] for _ in range(tokens)]).astype(np.int32)
    wts = rng.random((tokens, 2)).astype(np.float32)
    x = rng.standard_normal((tokens, hid)).astype(np.float32)
    s, eids, post = o.moe_align_block_size(ids, 32, e)
    x *= 4.0 / np.abs(o.moe_a8(x, w13, s, eids, post, t13, 2 * inner, 2, tokens, 32)).max()
    return [torch.from_numpy(x).to(dtype).cuda(), *(torch.from_numpy(a).cuda() for a in (w13, w2, wts, ids))]


# 16-bit layers, against the kernels behind these (a workspace off 16 bytes): K of the second product in one part and in several,
# an output that takes no stores of four or eight values
@pytest.mark.parametrize("dtype", (torch.float16, torch.bfloat16))
@pytest.mark.parametrize("t13,t2,tokens,e,hid,inner,n_out", [
    (o.Q4_K, o.Q6_K, 150, 4, 768, 2048, 768), (o.Q4_0, o.Q4_0, 200, 5, 256, 1024, 1028), (o.Q8_0, o.Q4_0, 150, 4, 512, 1792, 512),
    (o.Q5_K, o.Q8_0, 130, 4, 256, 1536, 250), (o.Q6_K, o.Q5_K, 150, 4, 256, 1536, 264)])
def test_moe_layer_16_bit(t13, t2, tokens, e, hid, inner, n_out, dtype):
    from vllm_gguf_plugin_prism_amd import _lib
    assert _lib.lib().gguf_moe_mmq_layer_wide(t13, t2, hid, inner, n_out, 2, tokens, e) == 1
    args = layer_inputs(np.random.default_rng(inner + n_out), t13, t2, tokens, e, hid, inner, dtype, n_out)
    got, want = (layer("gguf_moe_mmq_layer", *args, t13, t2, off).float().cpu().numpy() for off in (0, 8))
    # (the same roundings; a sum whose last bit differs may round to the neighbouring 16-bit value, of the result or of h)
    assert np.isfinite(want).all() and o.rel_l2(got, want) <= {torch.float16: 1e-3, torch.bfloat16: 4e-3}[dtype]


# the kernels that fetch rows in pieces of 16 bytes (wide tiles; streaming tiles at 16 and at 32 slots a block, and with the
# per-pair operator's arithmetic) leave a workspace off that boundary to the others
@pytest.mark.parametrize("entry,t13,t2,tokens,e,hid,inner", [
    ("gguf_moe_mmq_layer", o.Q4_K, o.Q6_K, 200, 5, 256, 1024), ("gguf_moe_mmq_layer", o.Q4_0, o.Q4_0, 200, 5, 256, 1024),
    ("gguf_moe_mmq_layer", o.Q4_0, o.Q8_0, 70, 16, 512, 768), ("gguf_moe_mmq_layer", o.Q4_0, o.Q4_0, 80, 8, 256, 256),
    ("gguf_moe_vec_layer", o.Q4_K, o.Q4_K, 48, 16, 512, 768)])
def test_layers_with_a_workspace_off_16_bytes(entry, t13, t2, tokens, e, hid, inner):
    rng = np.random.default_rng(tokens + inner)
    args = layer_inputs(rng, t13, t2, tokens, e, hid, inner, torch.float32)
    want = layer(entry, *args, t13, t2)
    for off in (8, 4):
        got = layer(entry, *args, t13, t2, off)
        # (two kernels: a quant of h may move by a step where the activation's last bit differs)
        assert o.rel_l2(got.cpu().numpy(), want.cpu().numpy()) <= 1e-3


# the same for the operators by themselves, on blocks of 16 slots
def test_expert_products_with_a_workspace_off_16_bytes():
    from vllm_gguf_plugin_prism_amd import _lib, ops
    L = _lib.lib()
    rng = np.random.default_rng(16)
    t, e, k, n = 40, 8, 512, 256
    w = torch.from_numpy(np.stack([o.make_weights(rng, o.Q4_K, n, k) for _ in range(e)])).cuda()
    x = torch.from_numpy(rng.standard_normal((t, k)).astype(np.float32)).cuda()
    ids = torch.from_numpy(np.stack([rng.permutation(e)[:2] for _ in range(t)]).astype(np.int32)).cuda()
    sorted_ids, experts, post = ops.moe_align_block_size(ids, 16, e)
    stream = torch.cuda.current_stream().cuda_stream
    nbytes = L.gguf_moe_vec_workspace_bytes(t, 2, k, e)
    got = {}
    for off in (0, 8, 4):
        ws = torch.empty(nbytes + 32, dtype=torch.uint8, device="cuda")
        a, b = (torch.empty(2 * t, n, dtype=torch.float32, device="cuda") for _ in range(2))
        assert L.gguf_moe_vec_act(x.data_ptr(), 0, ws.data_ptr() + off, w.data_ptr(), ids.data_ptr(), a.data_ptr(), o.Q4_K, n, k, 2, t, 0, e, nbytes, stream) == 0
        assert L.gguf_moe_mmq_block(x.data_ptr(), 0, ws.data_ptr() + off, w.data_ptr(), w.stride(0), sorted_ids.data_ptr(), experts.data_ptr(), post.data_ptr(),
                                    sorted_ids.numel(), b.data_ptr(), o.Q4_K, n, k, 2, t, 0, 16, e, stream) == 0
        got[off] = [y.cpu().numpy() for y in (a, b)]
    for off in (8, 4):
        for y, want in zip(got[off], got[0]):
            assert o.rel_l2(y, want) <= 1e-5


# a gate sum past the half-precision range on the negative side: the activation makes it not a number, and as a quant of h it is
# 0 on every route, so that a down format without an offset on the block's sum gives that token a row of numbers (the other
# route: a workspace off 16 bytes)
@pytest.mark.parametrize("t2", (o.Q6_K, o.Q8_0))
def test_a_gate_that_is_not_a_number(t2):
    from vllm_gguf_plugin_prism_amd import _lib
    rng = np.random.default_rng(t2)
    tokens, e, hid, inner, at = 150, 4, 512, 1792, 5
    assert _lib.lib().gguf_moe_mmq_layer_wide(o.Q8_0, t2, hid, inner, hid, 2, tokens, e) == 1
    x, w13, w2, wts, ids = layer_inputs(rng, o.Q8_0, t2, tokens, e, hid, inner, torch.float16)
    size = float(x.abs().max())
    x[:, :32] = 0.0                                         # (the first block: for that token and feature 3 alone)
    x[at, :32] = size
    row = w13.view(e, 2 * inner, hid // 32, 34)[:, 3]
    row.zero_()
    row[:, 0, :2] = torch.from_numpy(np.frombuffer(np.float16(200 / size).tobytes(), np.uint8).copy()).cuda()
    row[:, 0, 2:] = 0x81                                    # -127 * 32 * 200 = -812800
    want = layer("gguf_moe_mmq_layer", x, w13, w2, wts, ids, o.Q8_0, t2, 8)
    got = layer("gguf_moe_mmq_layer", x, w13, w2, wts, ids, o.Q8_0, t2)
    assert torch.isfinite(want).all() and torch.isfinite(got).all()
    assert o.rel_l2(got.float().cpu().numpy(), want.float().cpu().numpy()) <= 1e-3
    assert o.rel_l2(got[at].float().cpu().numpy(), want[at].float().cpu().numpy()) <= 1e-3
