"""Products of 17 to 64 rows whose operands stream through LDS (csrc/gemm_stream.hip) against 64 bits: at the edges of the tiles of
16 rows of A, for every count of weight tiles a workgroup takes, with fewer stages of k than are on their way at once, with
short last ranges of k, and through every epilogue."""

import pytest
import torch

from paged_attention_engine_amd.kernels import lib as K
from tests.plain import qwen2_plain as plain

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
# (N, K, k ranges): by the rule, 2 to 10 tiles a workgroup
SIZES = [(3080, 64, 1), (6144, 128, 1), (9728, 320, 1), (17936, 192, 1), (22024, 256, 1), (37888, 192, 1), (65552, 64, 1), (40, 1536, 3),
         (1536, 2240, 5), (4608, 704, 3), (5120, 1344, 6)]


@pytest.mark.parametrize("M", [17, 31, 32, 33, 48, 49, 64])
@pytest.mark.parametrize("N,K_,splits", SIZES)
def test_streamed_products(M, N, K_, splits):
    gen = torch.Generator(device=DEV).manual_seed(M + N)
    randn = lambda *shape: torch.randn(shape, generator=gen, device=DEV)
    a, w = randn(M, K_ + 8).bfloat16()[:, :K_], (randn(N, K_) * K_ ** -0.5).bfloat16()
    want = a.double() @ w.double().t()
    # float32 sums of products of bfloat16 numbers: as many roundings as terms, each of up to 2^-24 of the terms' sizes; random, so their root
    bound = 2.0 ** -24 * 8 * (a.double().pow(2) @ w.double().pow(2).t()).sqrt() * K_ ** 0.5 / 4 + 1e-6
    parts = torch.full((splits, M, N), float("nan"), device=DEV)
    K.gemm_skinny(parts, a, w, None, K.EPI_F32, splits)
    assert ((parts.double().sum(0) - want).abs() <= bound).all()
    b = randn(N).bfloat16()
    out = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=DEV)
    K.gemm_skinny(out, a, w, b, K.EPI_BF16, splits)
    full = want + b.double()
    assert ((out.double() - full).abs() <= 2.0 ** -8 * full.abs() + bound).all()
    # rows that are still to be divided by their root mean square
    shares = torch.rand(M, K.stat_tiles(K_), generator=gen, device=DEV)
    scale = (shares.double().sum(1) / K_ + 1e-6).rsqrt()[:, None]
    K.gemm_skinny(out, a, w, None, K.EPI_BF16, splits, row_scale=(shares, 1e-6))
    assert ((out.double() - want * scale).abs() <= 2.0 ** -8 * (want * scale).abs() + bound * scale * 2 + 1e-5).all()
    # into the residual, with the next product's rows
    residual, weight = randn(M, N), randn(N).bfloat16()
    rows = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=DEV)
    stats = torch.full((M, K.stat_tiles(N)), float("nan"), device=DEV)
    after = residual.clone()
    K.gemm_skinny(after, a, w, None, K.EPI_RESIDUAL, splits, following=(rows, weight, stats))
    assert ((after.double() - residual.double() - want).abs() <= bound + 2.0 ** -23 * after.double().abs()).all()
    assert torch.equal(rows, (after * weight.float()).bfloat16())
    assert torch.allclose(stats.double().sum(1), after.double().pow(2).sum(1), rtol=2e-6)
    if N % 16 == 0:  # blocks of 8 gate rows and their 8 others
        gated = torch.full((M, N // 2), float("nan"), dtype=torch.bfloat16, device=DEV)
        K.gemm_skinny(gated, a, w, None, K.EPI_SWIGLU, splits)
        gate, up = want.view(M, -1, 2, 8).unbind(2)
        exact = (torch.nn.functional.silu(gate) * up).reshape(M, -1)
        assert ((gated.double() - exact).abs() <= 2.0 ** -8 * exact.abs() + 4e-6 * (1 + gate.abs() + up.abs()).reshape(M, -1) ** 2 + 1e-6).all()
    K.check_tickets_zero(DEV)


@pytest.mark.parametrize("M", [17, 33, 64])
@pytest.mark.parametrize("N,K_,splits", [(1288, 1536, 3), (1272, 3584, 5), (16, 281344, 8), (1272, 1536, 3)])
def test_streamed_products_of_few_weight_rows(M, N, K_, splits):
    """At the line between few weight rows that are streamed and those that are not; ranges as they are cut, the last one shorter."""
    test_streamed_products(M, N, K_, splits)


@pytest.mark.parametrize("M", [17, 33, 64])
@pytest.mark.parametrize("nh,nkv,hd,rot,splits", [(28, 4, 128, 128, 3), (36, 8, 80, 32, 1), (50, 4, 96, 96, 1), (12, 2, 128, 64, 2)])
def test_streamed_projections_rotate_and_store(M, nh, nkv, hd, rot, splits):
    width, bs, N = 640, 16, (nh + 2 * nkv) * hd
    gen = torch.Generator().manual_seed(M + nh)
    a, w = torch.randn(M, width, generator=gen).bfloat16(), (torch.randn(N, width, generator=gen) * width ** -0.5).bfloat16()
    b = torch.randn(N, generator=gen).bfloat16()
    positions, tables = torch.arange(3, 3 + 5 * M, 5, dtype=torch.int32), torch.randperm(M * 25, generator=gen).int().view(M, 25)
    inv = K.rope_table(positions.to(DEV), plain.rope_inv_freq(rot, 1e4).to(DEV))
    pools = [torch.zeros(M * 25, nkv, *shape, dtype=torch.bfloat16, device=DEV) for shape in ((bs, hd), (hd, bs))]
    q = torch.empty(M, nh * hd, dtype=torch.bfloat16, device=DEV)
    K.gemm_skinny_rope(q, a.to(DEV), w.to(DEV), b.to(DEV), nh, nkv, hd, rot, inv, positions.to(DEV), torch.arange(M, dtype=torch.int32, device=DEV),
                       tables.to(DEV), bs, *pools, splits)
    x = (a.double() @ w.double().t() + b.double()).bfloat16().double().view(M, -1, hd)
    turned = x.clone()
    cos, sin = plain.rope_cos_sin(plain.rope_inv_freq(rot, 1e4, torch.float64), positions, torch.float64)
    turned[..., :rot] = x[..., :rot] * cos[:, None] + plain.rotate_half(x[..., :rot]) * sin[:, None]
    # a rounding of the projection, which may fall the other way (2^-7 of it), of each of a rotated pair, and of the result
    bound = 2.0 ** -7 * (x.abs().amax(-1, keepdim=True) * 1.5 + 0.01)
    assert ((q.double().cpu().view(M, nh, hd) - turned[:, :nh]).abs() <= bound[:, :nh]).all()
    for m in range(M):
        page, at = int(tables[m, int(positions[m]) // bs]), int(positions[m]) % bs
        assert ((pools[0][page, :, at].double().cpu() - turned[m, nh:nh + nkv]).abs() <= bound[m, nh:nh + nkv]).all()
        assert ((pools[1][page, :, :, at].double().cpu() - x[m, nh + nkv:]).abs() <= bound[m, nh + nkv:]).all()
