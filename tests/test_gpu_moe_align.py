"""The routing sort (csrc/moe_aux.hip) where its parts meet: ids in registers and behind them, blocks that are no power of two, experts without pairs."""
import numpy as np
import pytest
import torch

from oracle import gguf_oracle as o

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("numel,experts,block", [(1, 1, 1), (64, 3, 7), (4096, 128, 32), (4097, 129, 32), (9001, 64, 48), (70000, 8, 16), (2400, 1024, 16), (63, 200, 64)])
def test_whole_result(numel, experts, block):
    from vllm_gguf_plugin_prism_amd import _lib
    rng = np.random.default_rng(numel)
    ids = (rng.integers(0, experts + 1, numel) ** 2 // max(experts, 1)).astype(np.int32)   # uneven; a few name no expert
    want, want_e, want_n = o.moe_align_block_size(ids[:, None], block, experts)
    cap = numel + experts * (block - 1)
    blocks = (cap + block - 1) // block + 3
    s, e, n = (torch.full((k,), -7, dtype=torch.int32, device="cuda") for k in (cap + 5, blocks, 1))
    assert _lib.lib().gguf_moe_align_block_size(torch.from_numpy(ids).cuda().data_ptr(), numel, experts, block, s.data_ptr(), cap, e.data_ptr(), blocks, n.data_ptr(),
                                                torch.cuda.current_stream().cuda_stream) == 0
    total = int(np.asarray(want_n).reshape(-1)[0])
    s, e = s.cpu().numpy(), e.cpu().numpy()
    assert n.item() == total and (s[:total] == np.asarray(want)[:total]).all() and (s[total:cap] == numel).all() and (s[cap:] == -7).all()
    assert (e[:total // block] == np.asarray(want_e)[:total // block]).all() and (e[total // block:] == -1).all()
