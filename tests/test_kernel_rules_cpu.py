"""The rules by which the kernel library chooses a route for a call, and the memory it asks for: plain host code, asked here
without a GPU."""

import torch

from paged_attention_engine_amd.kernels import lib as K


def test_routers_that_one_workgroup_reads_are_small():
    pays = lambda dtype, n, k: bool(K.library().pae_moe_choose_pays(K.code_of(dtype), n, k))
    assert pays(torch.bfloat16, 32, 1536) and pays(torch.bfloat16, 33, 1536) and pays(torch.bfloat16, 40, 2560)
    for n, k in ((64, 2048), (128, 2048), (256, 256), (256, 7168), (1024, 4096), (8, 7168)):
        assert not pays(torch.bfloat16, n, k) and not pays(torch.float32, n, k)


def test_large_tiles_of_experts_are_counted_in_fifteen_bits():
    """An expert may be named by every pair: its tiles of 128 rows, and the places of rows and weights in 32 bits."""
    rows = K.library().pae_moe_tile_rows
    assert [rows(n, 1536, 2240, 3072) for n in (512, 513, 4096, 4097, 12004)] == [16, 64, 64, 128, 128]
    assert rows(0x7fff * 128, 64, 64, 128) == 128 and rows(0x7fff * 128 + 1, 64, 64, 128) == 64
    assert rows(1 << 20, 4096, 2240, 8192) == 64 and rows(8192, 1536, 2240 + 32, 3072) == 64
