"""Which products the walking codebook GEMM (csrc/dense_walk_core.h) takes, and what the compiler gave it (no GPU needed)."""
import pytest

from test_kernel_resources import kernels
from vllm_gguf_plugin_prism_amd import _lib, ops

IQ4_XS, IQ3_S = 23, 21


# measured, us, dense_kernel / walked
@pytest.mark.parametrize("qt,m,n,k,plan", [
    (IQ4_XS, 17, 5120, 5120, (17, 8)), (IQ4_XS, 64, 4096, 4096, (1, 8)), (IQ4_XS, 256, 5120, 5120, (3, 4)),        # 17.5 / 11.0 (as they lie), 19.2 / 11.6, 32.4 / 30 to 32
    (IQ3_S, 141, 4160, 18688, (0, 0)), (IQ4_XS, 512, 5120, 5120, (0, 0)), (IQ4_XS, 17, 1024, 4096, (0, 0)),       # 69 / 88, 52.5 / 52.3, 9.4 / 11.0
    (IQ4_XS, 4, 5120, 5120, (0, 0)), (IQ4_XS, 1025, 5120, 512, (0, 0))])                                         # not measured
def test_the_faster_kernel_is_taken(qt, m, n, k, plan):
    L = _lib.lib()
    qk, size = ops.quant_sizes(qt)
    assert divmod(L.gguf_dense_linear_walk(qt, n, k, m, k // qk * size, L.gguf_dense_linear_workspace_bytes(n, k, m)), 16) == plan


def test_a_workspace_without_room_is_not_taken():
    L, m, n, k, pitch = _lib.lib(), 33, 4096, 4096, 4096 // 256 * 136
    rows = 64 * k * 2
    assert L.gguf_dense_linear_workspace_bytes(n, k, m) >= rows
    assert L.gguf_dense_linear_walk(IQ4_XS, n, k, m, pitch, rows) and L.gguf_dense_linear_walk(IQ4_XS, n, k, m, pitch, rows - 1) == 0


def test_nothing_goes_to_scratch():
    of = {name: n for name, n in kernels(_lib.LIB_PATH.read_bytes()) if "17dense_walk_kernelI" in name}
    assert of and not any(of.values())
