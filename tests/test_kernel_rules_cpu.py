"""The rules by which the kernel library chooses a route for a call, and the memory it asks for: plain host code, asked here
without a GPU."""

import ctypes
import os
import re

import pytest
import torch

from paged_attention_engine_amd.kernels import build
from paged_attention_engine_amd.kernels import lib as K


def part_of(M, N, K_, shared=True):
    part = (ctypes.c_int * 2)()
    K.library().pae_gemm_plain_part(M, N, K_, int(shared), ctypes.addressof(part))
    return tuple(part)


@pytest.mark.parametrize("M,N,K_", [(200, 3584, 18944), (601, 3584, 18944), (800, 3584, 18944), (601, 2048, 11008), (2000, 512, 18944),
                                    (3000, 512, 18944), (24000, 64, 18944), (65, 24000, 18944), (64, 8000, 53248), (100, 100, 2000000)])
def test_memory_for_the_sums_of_shared_products_is_bounded(M, N, K_):
    """At most 128 MiB, or one row or column of tiles where its sums are more than that; every part of the product fits it."""
    blocks, (rows, cols) = -(-K_ // 512), part_of(M, N, K_)
    floats = K.library().pae_gemm_plain_scratch(M, N, K_)
    assert floats <= max(32 << 20, blocks * 64 * min(M, N))
    assert 0 < rows <= M and 0 < cols <= N and (rows == M or rows % 64 == 0) and (cols == N or cols % 64 == 0)
    assert floats in (0, blocks * rows * cols)


@pytest.mark.parametrize("M,N,K_", [(4194240, 16448, 1), (4194240, 4096, 64), (70000, 1 << 20, 1), (1, 1 << 30, 4), (64, 2000000000, 1)])
@pytest.mark.parametrize("shared", [False, True])
def test_products_of_any_size_fit_a_grid(M, N, K_, shared):
    """A grid's threads along x are counted in 32 bits: up to 512 a tile of 64 x 64, up to 768 a sixteen of columns of few rows."""
    rows, cols = part_of(M, N, K_, shared)
    assert 0 < rows <= M and 0 < cols <= N
    assert (-(-rows // 64) * -(-cols // 64) * 512 if rows > 64 else -(-cols // 16) * 768) < 1 << 32


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


def test_a_product_of_no_rows_is_done_whatever_its_types():
    for pair in ((0, 0), (1, 1), (1, 0), (0, 1)):
        assert K.library().pae_gemm_plain_shared(*pair, None, 8, 0, None, 8, 0, None, 0, None, 0, 0, 8, 8, 1, None, None) == 0


@pytest.mark.parametrize("M,N,K_", [(65, 896, 4864), (513, 896, 4864), (300, 256, 4096), (2048, 256, 4096), (65, 16, 8192), (4096, 64, 4096)])
def test_products_of_few_tiles_and_much_of_k_go_to_the_library(M, N, K_):
    """One chain of stages a tile takes longer there than the library's shares of k (1.2 to 2.7 times, with half the units idle or more); an
    activation, or sums of ranges of k for a caller that adds them, are still made here, and so is what has less of k or more tiles."""
    plan = K.library().pae_gemm_wide_plan
    assert plan(K.WIDE_PLAIN, -1, M, N, K_, 0) == -1
    assert plan(K.WIDE_PLAIN, 0, M, N, K_, 0) >= 0 and plan(K.WIDE_SUMS, -1, M, N, K_, 1) >> 8 >= 1
    assert plan(K.WIDE_PLAIN, -1, M, N, 2240, 0) >= 0 and plan(K.WIDE_PLAIN, -1, 150, 4608, 3584, 0) >= 0


def test_the_shape_of_a_product_between_one_and_two_small_tiles_a_unit():
    """Rows of 2,048 numbers and more come slower to two workgroups a unit: 128 x 96 is ahead of 64 x 128 there (24.8 against 28.1 us)."""
    assert K.library().pae_gemm_wide_plan(K.WIDE_PLAIN, -1, 300, 4608, 3584, 0) == 3 | 1 << 8


def test_products_of_many_rows_take_the_operands_that_the_library_takes():
    """Tensors that are not the GPU's, and shapes that do not fit each other, are the library's, to work on or to refuse."""
    from paged_attention_engine_amd.parts.linear import Linear

    a, w, bias = (torch.randn(*shape).to(torch.bfloat16) for shape in ((70, 128), (64, 128), (64,)))
    assert torch.equal(Linear(w)(a), torch.mm(a, w.t()))
    assert torch.equal(Linear(w, bias)(a), torch.addmm(bias, a, w.t()))
    for wrong in (a[:, :64].contiguous(), a[:, 0], a[None]):
        with pytest.raises(RuntimeError):
            Linear(w)(wrong)


def test_runs_of_a_prompt_choose_a_kernel_that_is_built_for_them():
    """Heads, pages and run counts of any size get an answer, and other widths and pages the kernel for any shape."""
    route = K.library().pae_attn_prefill_route
    assert [route(12, 128, 128, 16, -(-n // 128), n, -(-n // 16), 0) for n in (2, 128, 512, 2048, 8192)] == [0, 0, 0, 2, 4]
    assert route(12, 192, 128, 16, 42, 5000, 60, 0) == 4 and route(12, 192, 128, 16, 1, 128, 8, 0) == 0
    for n in (2, 600, 5000, 1 << 22):
        assert route(14, 64, 64, 16, -(-n // 128), n, -(-n // 16), 0) in (0, 2)
        for hd, vd, bs in ((96, 96, 16), (256, 256, 16), (128, 128, 32), (64, 64, 48), (128, 64, 16), (256, 128, 16)):
            assert route(12, hd, vd, bs, -(-n // 128), n, -(-n // bs), 0) == 0
        for window in (0, 1, 64, 4096):
            assert route(1, 128, 128, 16, -(-n // 128), n, 1 << 20, window) in (0, 2, 4)


@pytest.mark.parametrize("M", [17, 32, 33, 64])
def test_ranges_of_streamed_products_fit_their_scratch(M):
    """Ranges of whole stages that cover k, and room for the sums of whichever count of weight tiles a workgroup takes."""
    lib = K.library()
    for N in (16, 896, 1536, 3072, 3080, 4608, 10240, 37888, 131072):
        for k in (64, 896, 1536, 8960, 18944):
            ranges = lib.pae_stream_ranges(M, N, k)
            if not ranges:
                continue
            per = -(-(-(-k // ranges)) // 128) * 128
            assert 1 <= ranges <= 8 and per * (ranges - 1) < k and (ranges > 1 or N > 3072)
            floats, slots = lib.pae_skinny_ticket_floats(M, N, ranges), lib.pae_skinny_ticket_slots(M, N)
            for tiles in (2, 3, 4, 5, 6, 8, 10) if M > 32 else (2, 4, 6, 8, 10):
                groups, mine = -(-N // (16 * tiles)), -(-(tiles if M > 32 else tiles // 2) // 2)
                assert groups * 8 <= max(slots, 8) and groups * 8 * mine * ranges * 256 <= floats
    assert [lib.pae_stream_ranges(m, 4608, k) for m, k in ((16, 3584), (65, 3584), (64, 3592))] == [0, 0, 0]


@pytest.mark.parametrize("T,nh,nkv,hd,vd,blocks,bs", [(1, 12, 2, 128, 128, 64, 16), (64, 12, 2, 128, 128, 64, 16), (65, 12, 2, 128, 128, 64, 16),
                                                      (3, 40, 1, 64, 64, 5, 16), (8, 16, 16, 64, 200, 3, 64), (43, 12, 12, 64, 64, 64, 16),
                                                      (64, 16, 16, 64, 64, 64, 16), (520, 1, 1, 64, 64, 64, 16), (100, 16, 8, 64, 64, 64, 16),
                                                      (9, 80, 1, 64, 64, 64, 16), (1, 1, 1, 4, 4, 8, 16), (2, 8, 2, 256, 256, 6000, 16)])
def test_scratch_of_shared_out_chunks(T, nh, nkv, hd, vd, blocks, bs):
    """Every chunk's sums have room, within 64 MiB; what is not asked of the library has none; other types and pools use none."""
    scratch = lambda *args: K.library().pae_paged_attention_scratch(*args)
    floats, chunks = scratch(0, 256, 512, blocks, bs, T, nh, nkv, hd, vd, 0), -(-blocks * bs // 64)
    assert floats in (0, T * nh * chunks * (vd + 2)) and floats <= 16 << 20
    if T * nkv > K.ATTENTION_SPLIT_GROUPS or blocks * bs <= 128:
        assert floats == 0
    assert scratch(1, 256, 512, blocks, bs, T, nh, nkv, hd, vd, 0) == scratch(0, 260, 512, blocks, bs, T, nh, nkv, hd, vd, 0) == 0
    assert scratch(0, 256, None, blocks, bs, T, nh, 1, hd, vd, 1) == 0
    assert K.library().pae_paged_attention_scratch(0, 256, 512, 64, 16, 3, 12, 2, 128, 128, 0) == 3 * 12 * 16 * 130


@pytest.mark.parametrize("T,S,D", [(1, 1, 128), (160, 1, 128), (319, 2, 64), (320, 2, 64), (320, 1, 32), (4000, 16, 256), (200, 1, 130), (500, 1, 260)])
def test_scratch_of_linear_attention_by_chunks(T, S, D):
    """Where a step goes by chunks, whatever its sequences, the scratch of its tokens has room for 16 factors a token and head."""
    lib, H, V = K.library(), 3, 40
    part = lambda n: -(-n // 4) * 4
    rows = 3 * part(T * H * D) + 2 * part(T * H * V)
    need = rows + part(T * H * (16 if lib.pae_linear_attention_by_chunks(T, S, D) else 1))
    assert lib.pae_linear_attention_work_floats(T, H, D, V) >= need
    assert not lib.pae_linear_attention_by_chunks(64, 64, D)


def test_the_plain_entry_of_wide_products_refuses_rotated_heads():
    """Mode 3 needs the heads' sizes and pools, which its own entry point brings; the places behind the operands are never read."""
    lib = K.library()
    plan = lib.pae_gemm_wide_plan(K.WIDE_GATED, -1, 128, 256, 128, 0)
    assert lib.pae_gemm_wide(3, -1, plan, 1 << 20, 256, 1 << 20, 128, 1 << 20, None, 0, 128, 256, 128, None) != 0
    assert "entry point of their own" in lib.pae_last_error().decode()
    for hd in (0, 32, 80):
        assert lib.pae_gemm_wide_rope(plan, 1 << 20, 256, 1 << 20, 128, 1 << 20, None, 0, 128, 128, 2, 0, hd, 0, None, None, None, None, 0, 16, None, None, None) != 0


@pytest.mark.parametrize("M,N,k,ranges", [(64, 4608, 3592, 3), (64, 37888, 3592, 3), (48, 37888, 3592, 2), (33, 10240, 18952, 3), (64, 17920, 1544, 1),
                                          (64, 16384, 1544, 3), (32, 16384, 1544, 3), (31, 16384, 1544, 1), (64, 2048, 3592, 1), (16, 4608, 3592, 1)])
def test_ranges_of_products_that_are_not_streamed(M, N, k, ranges):
    """k that is no multiple of 64, and weights off 16 bytes, which leave the streamed products' ranges to the other kernels' own rule."""
    assert K.whole_sum_splits(N, k, M) == ranges
    off = torch.empty(8, dtype=torch.bfloat16)[1:]
    assert off.data_ptr() % 16
    assert K.whole_sum_splits(N, k // 64 * 64, M, off) == K.whole_sum_splits(N, k // 64 * 64 + 8, M)
    assert K.skinny_splits(N, k, M, off) == K.skinny_splits(N, k, M) and K.residual_splits(2048, k, M, off) == K.residual_splits(2048, k, M)
    streamed = K.library().pae_stream_ranges(M, 4608, 3584)
    assert K.whole_sum_splits(4608, 3584, M) == (streamed or 1)


def test_rules_of_sizes_are_worked_out_once(monkeypatch):
    """A step that is not recorded asks them for every product of every layer, and the host bounds a short prompt's."""
    off = torch.empty(8, dtype=torch.bfloat16)[1:]
    asked = [(rule, N, k, M, w) for rule in (K.whole_sum_splits, K.residual_splits, K.skinny_splits) for M in (1, 16, 17, 40, 64)
             for N, k in ((2048, 1536), (37888, 3584), (3584, 18944), (4608, 3592)) for w in (None, off)]
    before = [rule(N, k, M, w) for rule, N, k, M, w in asked]
    monkeypatch.setattr(K, "library", None)
    monkeypatch.setattr(K, "_part_ranges", None)
    monkeypatch.setattr(K, "_whole_sum_ranges", None)
    assert [rule(N, k, M, w) for rule, N, k, M, w in asked] == before
    assert any(a != b for a, b in zip(before[0::2], before[1::2]))  # weights off 16 bytes have their own


def test_projections_that_the_library_is_ahead_at_are_not_rotated_in_tiles():
    """Few tiles with much of k, as for plain products, go to the library and a rotation behind it; elsewhere the tiles are those of gated products."""
    plan = K.library().pae_gemm_wide_plan
    for M, N, k in ((65, 1536, 8192), (127, 768, 4096), (240, 768, 4096), (993, 1536, 8192), (240, 5120, 6144), (127, 1280, 3072)):
        assert plan(K.WIDE_ROTATED, -1, M, N, k, 0) == plan(K.WIDE_PLAIN, -1, M, N, k, 0) == -1, (M, N, k)
    for M, N, k in ((65, 1152, 896), (2048, 2048, 1536), (2500, 2560, 2048), (993, 4608, 3584), (6030, 4608, 3584), (385, 7168, 5120), (300, 12288, 4096),
                    (6000, 1536, 8192), (700, 768, 4096), (70, 2048, 64)):
        assert plan(K.WIDE_ROTATED, -1, M, N, k, 0) == plan(K.WIDE_GATED, -1, M, N, k, 0) >= 0, (M, N, k)


def test_short_runs_beside_a_long_context_choose_by_their_own_keys():
    """The tables are as wide as the longest sequence of a step, which may bring a single token."""
    from paged_attention_engine_amd.parts.attention import most_keys
    from paged_attention_engine_amd.parts.base import StepContext

    step = lambda lens, past: StepContext(torch.bfloat16, torch.device("cpu"), sum(lens), len(lens), None, None, {}, None, None, q_lens=lens, past_lens=past)
    ctx = step([1, 128, 1, 40], [4000, 0, 9, 200])
    assert most_keys(ctx) == most_keys(ctx) == 240 and most_keys(step([1, 1], [70, 3])) == 0
    route = lambda runs, tokens, keys, nh=12: K.library().pae_attn_prefill_route(nh, 128, 128, 16, runs, tokens, -(-keys // 16), 0)
    assert route(2, 168, 240) == 0 and route(2, 168, 4001) == 2
    assert [route(n, 90 * n, 90) for n in (1, 5, 6)] == [0, 0, 2] and route(6, 360, 60) == 0 and route(3, 270, 90, 28) == 2


def test_products_of_one_workgroup_a_unit_that_are_ahead_are_not_streamed():
    """Workgroups of seven and eight wavefronts up to 48 rows, and beyond that with much of k; five and six where streaming would cut k
    often or k is long."""
    one = K.library().pae_one_workgroup_a_unit
    for M, N, k in ((17, 17920, 1536), (32, 22016, 2048), (33, 28672, 4096), (48, 27648, 5120), (64, 28672, 4096), (64, 32768, 8192), (48, 17920, 8192), (40, 28672, 1024),
                    (48, 21504, 5120)):
        assert one(M, N, k) and K.whole_sum_splits(N, k, M) == 1, (M, N, k)
    for M, N, k in ((16, 17920, 1536), (65, 28672, 4096), (33, 17920, 1536), (64, 17920, 1536), (64, 22016, 2048), (48, 24576, 3072), (64, 28672, 2048),
                    (64, 17920, 8192), (48, 17920, 4096), (32, 16384, 1536), (20, 37888, 3584)):
        assert not one(M, N, k), (M, N, k)
        assert M == 16 or M == 65 or K.whole_sum_splits(N, k, M) == K.library().pae_stream_ranges(M, N, k) > 0


@pytest.mark.parametrize("M", [17, 32, 48, 64])
def test_few_and_short_weight_rows_are_not_streamed(M):
    """A product whose weights are read in less time than a streamed product starts in keeps the ranges of the other kernels."""
    for N, k in ((640, 3072), (640, 6144), (896, 4864), (1024, 4096), (1280, 3072), (16, 65536)):
        assert K.library().pae_stream_ranges(M, N, k) == 0 and K.skinny_splits(N, k, M) == K.skinny_splits(N, k + 8, M), (N, k)
    for N, k in ((640, 12288), (1024, 6144), (1536, 2240), (1536, 8960), (1296, 3072)):
        assert K.library().pae_stream_ranges(M, N, k) > 1, (N, k)


@pytest.mark.parametrize("M", [16, 17, 32, 33, 64])
def test_ranges_of_partial_sums_cost_less_than_tickets(M):
    """Only where a streamed product would take one range; those cover k, and products that add themselves into the residual keep theirs."""
    lib = K.library()
    for N in (16, 640, 1536, 3072, 3088, 3584, 4096, 8192, 10240):
        for k in (64, 384, 768, 1536, 2048, 4096, 8960, 18944):
            one, part = lib.pae_stream_ranges(M, N, k), lib.pae_stream_part_ranges(M, N, k)
            assert part == one or (one == 1 and part <= 8 and (-(-(-(-k // part)) // 128) * 128) * (part - 1) < k and k // part >= 384), (N, k)
            if M > 16 and N > 3072:
                assert K.skinny_splits(N, k, M) == part and K.residual_splits(N, k, M) == one, (N, k)
    assert lib.pae_stream_part_ranges(32, 8192, 4096) > 1 == lib.pae_stream_ranges(32, 8192, 4096)


def test_the_polynomial_of_gelu_is_the_one_that_was_fitted():
    """exp(x^2) erfc(x) by the numbers in the source, in 64 bits, over all x whose GELU is not below float32's least: within 3e-7 of it,
    where a fit of its degree reaches 1.5e-8 and the numbers' own rounding leaves 1.4e-7."""
    with open(os.path.join(build.CSRC, "common.h")) as handle:
        body = re.search(r"float gelu_to_bf16\(float z\) \{(.*?)\n\}", handle.read(), re.S).group(1)
    number = r"(-?[\d.e-]+)f"
    slope = float(re.search(r"x = %s \* a" % number, body).group(1))
    q = [float(re.search(r"float q = %s;" % number, body).group(1))] + [float(c) for c in re.findall(r"q = fmaf\(q, s, %s\)" % number, body)]
    x = torch.linspace(0, 9.4, 100001, dtype=torch.float64)
    at = torch.tensor([slope, *q], dtype=torch.float32).double()  # as the kernels hold them
    s = at[0] * 2 ** 0.5 * x
    s = s / (1 + s)
    value = torch.zeros_like(x)
    for c in at[1:]:
        value = value * s + c
    assert len(q) == 9 and ((2 * (0.5 + s * value) / torch.special.erfcx(x) - 1).abs() < 3e-7).all()


def test_ranges_of_k_leave_a_decode_program_the_layers_that_it_took():
    """A program's LDS holds a range's activations: the down product of a layer whose gate product fits has ranges that fit too, up to eight of
    them, or four of wider ones."""
    fits = lambda k, splits: K.program_takes_product(16, k, splits)
    longest = max(k for k in range(128, 8192, 128) if fits(k, 1))
    assert K._program_range() == longest and fits(longest, 1) and not fits(longest + 128, 1)
    for hidden in range(64, longest + 1, 64):
        tiles = -(-hidden // 16)
        most = 4 if hidden > 3072 else min(8, 512 // tiles)
        for ff in {longest * most, longest * most - 8, 4 * hidden, 8 * hidden // 3 // 8 * 8, 5 * hidden, 8960}:
            if ff <= longest * most:
                assert fits(ff, K.residual_splits(hidden, ff, 16)), (hidden, ff)


@pytest.mark.parametrize("N,K_", [(896, 4864), (1536, 8960), (3200, 8640), (3584, 18944), (5120, 5120), (5120, 13824), (5120, 27648), (8192, 29568), (9216, 300)])
def test_ranges_of_few_rows_follow_from_the_weights_alone(N, K_):
    """Up to 16 rows a row's sums are the same bits whatever it is batched with; no range is empty."""
    for rule in (K.residual_splits, K.skinny_splits):
        ranges = {rule(N, K_, M) for M in range(1, 17)}
        assert len(ranges) == 1
        r = ranges.pop()
        assert 1 <= r <= 8 and (r - 1) * (-(-(-(-K_ // r)) // 128) * 128) < K_


def test_single_tokens_of_many_value_heads_a_key_head_take_one_launch_only_where_they_are_many():
    """A workgroup takes a key head's value heads one after another: few sequences of many value heads go by the separate kernels, whose heads run beside
    each other."""
    pays = lambda seqs, G, H: bool(K.library().pae_tokens_step_pays(seqs, G, H))
    assert all(pays(seqs, G, H) for seqs in (1, 8, 1000) for G, H in ((1, 1), (12, 12), (6, 12), (4, 16), (28, 28)))
    assert not any((pays(1, 1, 16), pays(64, 1, 16), pays(1, 2, 16), pays(8, 2, 16), pays(4, 4, 32), pays(32, 2, 28), pays(8, 1, 8)))
    assert all((pays(128, 1, 16), pays(32, 2, 16), pays(16, 4, 32), pays(64, 2, 28), pays(64, 1, 8), pays(60000, 1000, 64000)))
