"""The walking tile kernel (csrc/tile_walk_core.h) at the edges of its tiles, panels and bands, in every form that a linear layer's call may have, and
the kernels behind it where they still run, against the CPU oracle."""
import numpy as np
import pytest
import torch

from oracle import gguf_oracle as o

pytestmark = pytest.mark.gpu

BLOCKS = (o.Q4_0, o.Q5_0, o.Q8_0, o.Q4_K, o.Q5_K)   # a scale per 32 values
GROUPS = (o.Q6_K, o.Q3_K)                            # per 16
TYPES = BLOCKS + GROUPS
OLDER = (o.Q4_0, o.Q5_0, o.Q8_0)


def product(qtype, m, n, k, pad=0, offset=0, dt=torch.float32, column=0, spare=0, rows=np.s_[:], tolerance=1e-5, check=None):
    from vllm_gguf_plugin_prism_amd import dispatch
    rng = np.random.default_rng(n + m)
    packed = o.make_weights(rng, qtype, n, k)
    rb = packed.shape[1]
    if check:
        check(rb + pad)
    raw = torch.zeros(offset + n * (rb + pad), dtype=torch.uint8, device="cuda")
    w = raw[offset:].view(n, rb + pad)[:, :rb]
    w.copy_(torch.from_numpy(packed))
    x = torch.from_numpy(rng.standard_normal((m, k)).astype(np.float32) + 0.3).to(dt)
    bias = torch.from_numpy(rng.standard_normal(n).astype(np.float32)).to(dt)
    wide = torch.full((m, column + n + spare), 7.0, dtype=dt, device="cuda")
    out = wide[:, column:column + n]
    assert dispatch.fused_mul_mat_gguf(x.cuda(), w, qtype, out=out, bias=bias.cuda()) is out
    want = o.mul_mat_a8(packed, x[rows].float().numpy(), qtype, n, "mmq") + bias.float().numpy()
    assert o.rel_l2(out[rows].float().cpu().numpy(), want) <= tolerance
    assert bool((wide[:, :column] == 7).all()) and bool((wide[:, column + n:] == 7).all())


def walked(qtype, m, n, k, plan=None):
    from vllm_gguf_plugin_prism_amd import ops

    def check(pitch):
        got = ops._linear_walk(qtype, n, k, m, pitch)
        assert got == plan if plan else got[0]
    return check


def tall_cut(qtype, size):
    """Q8_0 has no tall tiles where a pitch moves its panels inside 16 bytes."""
    return qtype == o.Q8_0 and size[3] % 16 != 0 and size[4][0] > 2


# each height of tiles with each number of waves that it has: waves without a panel, with one, two and three; last tiles of rows and columns in part; rows of
# W a pitch apart that moves them through the positions inside 16 bytes
@pytest.mark.parametrize("qtype,m,n,k,pad,plan", [(q, *s) for q in BLOCKS for s in (
    (33, 323, 512, 0, (1, 4)), (67, 4148, 1280, 2, (1, 4)), (35, 308, 1280, 0, (1, 8)), (37, 332, 4352, 6, (1, 8)),
    (33, 8734, 512, 0, (2, 4)), (135, 3307, 2304, 14, (2, 4)), (36, 4317, 1280, 2, (2, 8)), (142, 1635, 5376, 0, (2, 8)),
    (65, 11337, 512, 6, (3, 4)), (332, 2814, 2304, 0, (3, 4)), (193, 5656, 1792, 10, (4, 4)), (591, 2387, 2304, 0, (4, 4))) if not tall_cut(q, s)] + [
    (o.Q8_0, 65, 11337, 512, 16, (3, 4)), (o.Q8_0, 193, 5656, 1792, 16, (4, 4)), (o.Q8_0, 65, 11337, 512, 6, (2, 4)), (o.Q8_0, 193, 5656, 1792, 10, (2, 4))] + [
    (q, *s) for q in GROUPS for s in (
    (35, 301, 512, 2, (1, 4)), (67, 4148, 1280, 4, (1, 4)), (33, 4267, 2560, 0, (1, 4)), (34, 305, 1280, 0, (1, 8)), (36, 325, 4352, 6, (1, 8)),
    (35, 8218, 512, 8, (2, 4)), (33, 8279, 1280, 10, (2, 4)), (36, 4123, 1280, 12, (2, 8)), (71, 8418, 1280, 14, (3, 4)))] + [
    (o.Q6_K, 135, 3307, 2304, 2, (2, 4)), (o.Q6_K, 142, 1635, 5376, 0, (2, 8)), (o.Q6_K, 135, 6029, 2304, 0, (3, 4)),
    (o.Q3_K, 97, 4257, 2304, 2, (2, 4)), (o.Q3_K, 104, 2174, 4352, 0, (2, 8)), (o.Q3_K, 202, 4241, 2304, 0, (3, 4)),
    (o.Q3_K, 98, 8309, 512, 0, (4, 4)), (o.Q3_K, 97, 8336, 1280, 6, (4, 4)), (o.Q3_K, 296, 4202, 2304, 14, (4, 4))])
def test_edges(qtype, m, n, k, pad, plan):
    product(qtype, m, n, k, pad, rows=np.r_[:3, m - 35:m], check=walked(qtype, m, n, k, plan))


# the last panel has one block, three, seven; one panel that is not whole
@pytest.mark.parametrize("qtype", OLDER)
@pytest.mark.parametrize("m,n,k,pad", [(70, 333, 1056, 0), (45, 333, 1120, 4), (130, 333, 2528, 0), (37, 333, 224, 2)])
def test_last_panels(qtype, m, n, k, pad):
    product(qtype, m, n, k, pad, check=walked(qtype, m, n, k))


# more rows than a band has: bands of one row block and of several, the last one with fewer of them
@pytest.mark.parametrize("qtype,m,n,k,plan,band,last", [(o.Q4_K, 300, 100, 9216, (1, 8), 9, 1), (o.Q8_0, 1351, 286, 2048, (2, 8), 21, 1), (o.Q4_K, 1715, 582, 2048, (3, 4), 14, 4),
                                                        (o.Q8_0, 1921, 772, 2048, (4, 4), 10, 6), (o.Q8_0, 261, 1909, 14592, (3, 4), 1, 1)])
def test_bands(qtype, m, n, k, plan, band, last):
    blocks = -(-m // (32 * plan[0]))
    fit = max(1, (3 << 20) // (plan[0] * -(-k // 256) * 9216))
    assert fit == band < blocks and blocks - (blocks - 1) // band * band == last
    at = 32 * plan[0] * band
    product(qtype, m, n, k, rows=np.r_[:3, at - 2:at + 2, m - 35:m], check=walked(qtype, m, n, k, plan))


# activations of every type, weights that begin anywhere, results that are columns of a wider tensor
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("offset,pad,column,spare", [(0, 0, 0, 0), (2, 14, 3, 4), (16, 16, 4, 4), (6, 4, 1, 0)])
@pytest.mark.parametrize("qtype", TYPES)
def test_forms(qtype, offset, pad, column, spare, dt):
    m, n, k = 67, 333, 2304
    # two roundings to 16 bits (product, product plus bias), each half a unit in the last place of 11 or 8 bits
    product(qtype, m, n, k, pad, offset, dt, column, spare, tolerance={torch.float32: 1e-5, torch.float16: 2.0 ** -10, torch.bfloat16: 2.0 ** -7}[dt],
            check=walked(qtype, m, n, k, (1, 8)))


# a value that is not a number stays in its row
def test_rows_do_not_meet():
    from vllm_gguf_plugin_prism_amd import ops
    m, n, k = 67, 333, 2304
    rng = np.random.default_rng(1)
    w = torch.from_numpy(o.make_weights(rng, o.Q4_K, n, k)).cuda()
    assert ops._linear_walk(o.Q4_K, n, k, m, w.shape[1])[0]
    x = torch.randn(m, k, device="cuda")
    y = ops.ggml_mul_mat_a8(w, x, o.Q4_K, n)
    x[40, 1000] = float("nan")
    z = ops.ggml_mul_mat_a8(w, x, o.Q4_K, n)
    assert bool(z[40].isnan().all()) and torch.equal(z[:40], y[:40]) and torch.equal(z[41:], y[41:])


# A block whose largest value is past 127 times a half's largest has an infinite scale (its sum of the inputs is finite here: the two large ones cancel): the result is an infinity of
# the sum's sign, no number where the sum is 0.  The rows beside it have the bits that they have without it.
@pytest.mark.parametrize("qtype,m,n,k,pad,plan", [(q, *s) for q in BLOCKS for s in ((35, 308, 1280, 0, (1, 8)), (135, 3307, 2304, 14, (2, 4)), (332, 2814, 2304, 0, (3, 4)), (591, 2387, 2304, 2, (4, 4))) if not tall_cut(q, s)] + [
    (q, 35, 301, 512, 2, (1, 4)) for q in GROUPS] + [(o.Q8_0, 591, 2387, 2304, 0, (4, 4))] + [(o.Q6_K, 142, 1635, 5376, 0, (2, 8)), (o.Q6_K, 135, 6029, 2304, 0, (3, 4)), (o.Q3_K, 202, 4241, 2304, 0, (3, 4)), (o.Q3_K, 296, 4202, 2304, 14, (4, 4))])
def test_infinite_block_scales(qtype, m, n, k, pad, plan):
    from vllm_gguf_plugin_prism_amd import ops
    rng = np.random.default_rng(n)
    packed = o.make_weights(rng, qtype, n, k)
    w = torch.zeros(n, packed.shape[1] + pad, dtype=torch.uint8, device="cuda")[:, :packed.shape[1]]
    w.copy_(torch.from_numpy(packed))
    assert ops._linear_walk(qtype, n, k, m, w.stride(0)) == plan
    x = rng.standard_normal((m, k)).astype(np.float32)
    without = ops.ggml_mul_mat_a8(w, torch.from_numpy(x).cuda(), qtype, n).cpu()
    places = {0: (0, 0, 17), 2: (k - 32, 3, 30), 5: (k // 64 * 32, 8, 9), 31: (256, 20, 1), m - 1: (k - 64, 31, 5)}   # row: block, places of the large values in it
    for row, (at, i, j) in places.items():
        x[row, at + i], x[row, at + j] = 3e9, -3e9
    got = ops.ggml_mul_mat_a8(w, torch.from_numpy(x).cuda(), qtype, n).cpu()
    rows = list(places)
    q, d8, s8 = o.quantize_q8_1(x[rows])
    wi, ws, _, group = o.unpack(packed, qtype)
    values = (np.repeat(ws, group, axis=1).astype(np.float64) * wi).reshape(n, k)   # (whole numbers of at most 36 bits times a half: exact)
    for r, (row, (at, _, _)) in enumerate(places.items()):
        assert np.isinf(d8[r, at // 32]) and np.isfinite(s8[r, at // 32])
        sums = values[:, at:at + 32] @ q[r, at:at + 32].astype(np.float64)
        want = torch.from_numpy(np.where(sums == 0, np.nan, np.copysign(np.inf, sums)))
        assert torch.equal(got[row].double().nan_to_num(0, 1, -1), want.nan_to_num(0, 1, -1)) and bool((got[row].isnan() == want.isnan()).all())
    others = [r for r in range(m) if r not in places]
    assert torch.equal(got[others], without[others])


# The kernels behind it at sizes where they still run: those whose estimate is shorter (few panels of many rows, few columns of long ones) ...
@pytest.mark.parametrize("qtype,m,n,k,route", [(o.Q4_0, 686, 2071, 320, 0), (o.Q4_0, 1782, 386, 256, 4), (o.Q5_0, 925, 552, 256, 0), (o.Q8_0, 1164, 539, 256, 0),
                                               (o.Q4_K, 717, 741, 256, 4), (o.Q4_K, 1007, 369, 9472, 2), (o.Q5_K, 1219, 569, 256, 4), (o.Q5_K, 822, 307, 14592, 2),
                                               (o.Q6_K, 66, 14616, 512, 0), (o.Q6_K, 633, 805, 256, 4), (o.Q6_K, 716, 306, 13056, 2), (o.Q3_K, 34, 23956, 256, 4),
                                               (o.Q3_K, 73, 16260, 256, 0)])
def test_kernels_of_what_is_not_walked(qtype, m, n, k, route):
    from vllm_gguf_plugin_prism_amd import ops

    def check(pitch):
        assert ops._linear_walk(qtype, n, k, m, pitch) == (0, 0) and ops._mmq_route(qtype, n, k, m, pitch) == route
    product(qtype, m, n, k, rows=np.r_[:3, m - 35:m], check=check)


# ... and with a workspace that has room for the quantized rows only: the streaming tiles, the int8 unit
@pytest.mark.parametrize("qtype", TYPES)
@pytest.mark.parametrize("m,n,k,route", [(40, 333, 1280, 1), (34, 8734, 4096, 0)])
def test_kernels_of_a_small_workspace(qtype, m, n, k, route):
    from vllm_gguf_plugin_prism_amd import _lib
    L = _lib.lib()
    rng = np.random.default_rng(n)
    packed = o.make_weights(rng, qtype, n, k)
    size = m * L.gguf_q8_1_row_bytes(k)
    assert L.gguf_linear_walk(qtype, n, k, m, packed.shape[1], size) == 0 and L.gguf_mmq_layer_route(qtype, n, k, m, packed.shape[1], size) == route
    x = rng.standard_normal((m, k)).astype(np.float32)
    w, xd, y, ws = torch.from_numpy(packed).cuda(), torch.from_numpy(x).cuda(), torch.empty(m, n, device="cuda"), torch.empty(size, dtype=torch.uint8, device="cuda")
    _lib.check(L.gguf_mmq(w.data_ptr(), xd.data_ptr(), 0, ws.data_ptr(), y.data_ptr(), int(qtype), n, k, m, torch.cuda.current_stream().cuda_stream), "gguf_mmq")
    assert o.rel_l2(y.cpu().numpy(), o.mul_mat_a8(packed, x, qtype, n, "mmq")) <= 1e-5


# captured once, replayed on other activations with eager work in between
def test_replays_as_eager():
    from vllm_gguf_plugin_prism_amd import dispatch, ops
    m, n, k = 77, 2080, 4096
    wn = o.make_weights(np.random.default_rng(3), o.Q8_0, n, k)
    assert ops._linear_walk(o.Q8_0, n, k, m, wn.shape[1])[0]
    w = torch.from_numpy(wn).cuda()
    xs = [torch.randn(m, k, dtype=torch.bfloat16, device="cuda") for _ in range(4)]
    x = xs[0].clone()
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        dispatch.fused_mul_mat_gguf(x, w, o.Q8_0)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = dispatch.fused_mul_mat_gguf(x, w, o.Q8_0)
    for xi in xs:
        x.copy_(xi)
        eager = dispatch.fused_mul_mat_gguf(x, w, o.Q8_0).clone()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager)
