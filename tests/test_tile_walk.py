"""Which products the walking tile kernel (csrc/tile_walk_core.h) takes, and what the compiler gave it (no GPU needed)."""
import pytest

from test_kernel_resources import kernels
from vllm_gguf_plugin_prism_amd import _lib, ops

Q4_0, Q5_0, Q8_0, Q3_K, Q4_K, Q5_K, Q6_K, Q2_K = 2, 6, 8, 11, 12, 13, 14, 10


# measured, us, the kernels that run otherwise / walked
@pytest.mark.parametrize("qt,m,n,k,plan", [
    (Q8_0, 77, 14336, 4096, (3, 4)), (Q4_K, 64, 4096, 4096, (1, 8)), (Q4_K, 128, 4096, 4096, (2, 8)), (Q8_0, 64, 4096, 4096, (1, 8)),   # 38.7 / 26.5, 16.1 / 10.8, 24.9 / 13.2, 19.4 / 12.6
    (Q4_K, 1501, 25456, 512, (0, 0)), (Q4_K, 1319, 8368, 512, (0, 0)), (Q2_K, 64, 4096, 4096, (0, 0)),                                  # 91 / 137, 37 / 50, not a format of it
    (Q6_K, 64, 4096, 4096, (1, 8)), (Q6_K, 512, 18944, 3584, (0, 0)), (Q3_K, 512, 14336, 4096, (4, 4)),                                 # 20.4 / 13.6, 184 / 187, 128 / 98
    (Q6_K, 118, 4400, 3328, (0, 0)), (Q4_K, 143, 3504, 15872, (0, 0)),                                                                  # 25.1 / 30.8, 52.8 / 61.1
    (Q4_K, 32, 4096, 4096, (0, 0)), (Q4_K, 2049, 4096, 4096, (0, 0))])                                                                  # at most 32 rows; not measured
def test_the_faster_kernel_is_taken(qt, m, n, k, plan):
    qk, size = ops.quant_sizes(qt)
    assert ops._linear_walk(qt, n, k, m, k // qk * size) == plan


# rows of Q8_0 a pitch apart that moves the panels inside 16 bytes, as in a padded merged tensor: LDS then has room for one workgroup of tall tiles (84 / 135 and, on these tiles,
# 44 / 41; tiles of 96 rows 61)
@pytest.mark.parametrize("m,n,k,pitch,plan", [(593, 13696, 2304, 2448, (4, 4)), (593, 13696, 2304, 2454, (0, 0)), (356, 2208, 7424, 7890, (2, 4))])
def test_panels_that_begin_anywhere(m, n, k, pitch, plan):
    assert ops._linear_walk(Q8_0, n, k, m, pitch) == plan


# the records of 33 rows are those of 64: more than the quantized rows, which are the least that a workspace holds
def test_a_workspace_without_room_is_not_taken():
    L, m, n, k, pitch = _lib.lib(), 33, 4096, 4096, 4096 // 256 * 144
    records = 64 * k // 256 * 288
    assert records > m * L.gguf_q8_1_row_bytes(k) and L.gguf_mmq_layer_workspace_bytes(Q4_K, n, k, m, pitch) >= records
    assert ops._linear_walk(Q4_K, n, k, m, pitch, records)[0] and ops._linear_walk(Q4_K, n, k, m, pitch, records - 1) == (0, 0)


def test_nothing_goes_to_scratch():
    of = {name: n for name, n in kernels(_lib.LIB_PATH.read_bytes()) if "16tile_walk_kernelI" in name}
    assert of and not any(of.values())
