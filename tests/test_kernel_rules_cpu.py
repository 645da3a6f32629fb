"""The rules by which the kernel library chooses a route for a call, and the memory it asks for: plain host code, asked here
without a GPU."""

import torch

from paged_attention_engine_amd.kernels import lib as K


def test_routers_that_one_workgroup_reads_are_small():
    pays = lambda dtype, n, k: bool(K.library().pae_moe_choose_pays(K.code_of(dtype), n, k))
    assert pays(torch.bfloat16, 32, 1536) and pays(torch.bfloat16, 33, 1536) and pays(torch.bfloat16, 40, 2560)
    for n, k in ((64, 2048), (128, 2048), (256, 256), (256, 7168), (1024, 4096), (8, 7168)):
        assert not pays(torch.bfloat16, n, k) and not pays(torch.float32, n, k)
