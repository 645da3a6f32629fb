"""Products of up to 16 rows (gemm_rows_kernel.h): every way to share out weight rows and k (16 or 8 weight rows a workgroup, one range, two or
four side by side, tickets, partial sums), edges of tiles and of 128-wide steps, against float64; the shares of the sums of
squares by 16 and by 8 columns.  Outputs are sums of K products of numbers of about 0.5 and 0.1: float32 sums are within 4e-6 of the
largest, a bfloat16 output within 2^-8 of itself."""

import pytest
import torch

from paged_attention_engine_amd.kernels import lib as K

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def operands(M, N, K_, seed):
    gen = torch.Generator().manual_seed(seed)
    a = (torch.randn(M, K_, generator=gen) * 0.5).bfloat16()
    w = (torch.randn(N, K_, generator=gen) * 0.1).bfloat16()
    return a, w, a.double() @ w.double().t(), gen


@pytest.mark.parametrize("M", [1, 4, 5, 9, 13, 16])
@pytest.mark.parametrize("N,K_", [(8, 8), (24, 136), (1000, 1032), (72, 2048), (6400, 392), (10272, 264), (10272, 1544), (3344, 648), (2568, 2048), (9736, 1536), (4616, 2568)])
def test_plain_and_float32_sums(M, N, K_):
    """Also several ranges: tickets (bfloat16) and partial sums (float32)."""
    a, w, want, gen = operands(M, N, K_, M + N + K_)
    bias = torch.randn(N, generator=gen).bfloat16()
    top = float(want.abs().max())
    d_a, d_w = a.to(DEV), w.to(DEV)
    for ranges in {1, 2 if K_ > 128 else 1, 3 if K_ > 512 else 1}:
        out = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=DEV)
        K.gemm_skinny(out, d_a, d_w, bias.to(DEV), splits=ranges)
        exact = want + bias.double()
        assert ((out.cpu().double() - exact).abs() <= 2.0 ** -8 * exact.abs() + 4e-6 * top).all()
        sums = torch.full((ranges, M, N), float("nan"), device=DEV)
        K.gemm_skinny(sums if ranges > 1 else sums[0], d_a, d_w, None, K.EPI_F32, ranges)
        assert (sums.cpu().double().sum(0) - want).abs().max() <= 4e-6 * top
    K.check_tickets_zero(DEV)


@pytest.mark.parametrize("M", [1, 8, 11, 16])
@pytest.mark.parametrize("N,K_", [(16, 264), (4864 * 2, 896), (10256, 1544), (22016, 520)])
def test_gated_sums(M, N, K_):
    a, w, want, _ = operands(M, N, K_, M + N + K_)
    out = torch.full((M, N // 2), float("nan"), dtype=torch.bfloat16, device=DEV)
    K.gemm_skinny(out, a.to(DEV), w.to(DEV), None, K.EPI_SWIGLU)
    gate, up = want.view(M, -1, 2, 8).unbind(2)
    exact = (gate * torch.sigmoid(gate) * up).reshape(M, -1)
    assert ((out.cpu().double() - exact).abs() <= 2.0 ** -8 * exact.abs() + 2e-5 * float(want.abs().max())).all()


@pytest.mark.parametrize("M", [1, 6, 10, 16])
@pytest.mark.parametrize("fine", [False, True])
@pytest.mark.parametrize("N,K_,ranges", [(1536, 8960, 4), (1544, 1536, 2), (200, 1032, 2), (3584, 4096, 2), (72, 1800, 4), (1000, 264, 1), (40, 1544, 3)])
def test_residual_sums_and_their_shares(M, fine, N, K_, ranges):
    a, w, want, gen = operands(M, N, K_, M + N + K_)
    residual = torch.randn(M, N, generator=gen) * 2.0
    w_norm = (1 + 0.2 * torch.randn(N, generator=gen)).bfloat16()
    want = want + residual.double()
    tiles = K.stat_tiles(N)
    width = 8 if fine and K.fine_stat_tiles(N, M) > tiles else 16
    stats = torch.full((M, tiles * 16 // width), float("nan"), device=DEV)
    nxt = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=DEV)
    out = residual.to(DEV)
    K.gemm_skinny(out, a.to(DEV), w.to(DEV), None, K.EPI_RESIDUAL, ranges, following=(nxt, w_norm.to(DEV), stats))
    assert (out.cpu().double() - want).abs().max() <= 4e-6 * float(want.abs().max())
    assert torch.equal(nxt.cpu(), (out.cpu() * w_norm.float()).bfloat16())
    squares = torch.zeros(M, tiles * 16, dtype=torch.float64)
    squares[:, :N] = out.cpu().double().pow(2)
    assert torch.allclose(stats.cpu().double(), squares.view(M, -1, width).sum(-1), rtol=2e-6, atol=1e-12)
    # the rows' scale from either kind of shares
    rows = K.scaled_rows(nxt, stats, 1e-6)
    exact = nxt.cpu().double() * torch.rsqrt(squares.sum(1, keepdim=True) / N + 1e-6)
    assert ((rows.cpu().double() - exact).abs() <= 2.0 ** -8 * exact.abs() + 1e-30).all()
    K.check_tickets_zero(DEV)


@pytest.mark.parametrize("M", [1, 5, 12, 16])
def test_a_row_is_the_same_bits_in_either_share_of_weight_rows(M):
    """Shares by 16 columns make a workgroup take 16 weight rows, by 8 eight of them; four rows and fewer take eight where more take 16."""
    a, w, _, gen = operands(M, 1536, 2304, M)
    nxt = torch.empty(M, 1536, dtype=torch.bfloat16, device=DEV)
    got = []
    for ranges in (1, 2, 4):
        for tiles in (K.stat_tiles(1536), K.fine_stat_tiles(1536)):
            out = torch.zeros(M, 1536, device=DEV)
            K.gemm_skinny(out, a.to(DEV), w.to(DEV), None, K.EPI_RESIDUAL, ranges,
                          following=(nxt, torch.ones(1536, device=DEV), torch.empty(M, tiles, device=DEV)))
            got.append(out)
    assert torch.equal(got[0], got[1]) and torch.equal(got[2], got[3]) and torch.equal(got[4], got[5])
    _, many, _, _ = operands(1, 12000, 776, 5)
    a = a[:, :776].contiguous().to(DEV)
    alone, among = torch.empty(1, 12000, device=DEV), torch.empty(M, 12000, device=DEV)
    K.gemm_skinny(alone, a[M - 1:], many.to(DEV), None, K.EPI_F32)
    K.gemm_skinny(among, a, many.to(DEV), None, K.EPI_F32)
    assert torch.equal(alone[0], among[M - 1])


@pytest.mark.parametrize("M", [1, 8, 12, 16])
@pytest.mark.parametrize("N,K_,ranges", [(2048, 1536, 1), (2560, 2048, 1), (72, 896, 1), (9736, 1536, 1), (40, 1536, 3), (4616, 2560, 1), (1536, 1536, 2), (3584, 3584, 2), (1544, 8960, 4)])
def test_an_infinite_number_of_a_row_is_added_once(M, N, K_, ranges):
    """Steps that reach past a range of k multiply nothing there: what stands at the row's end, or in another range, does not come in as zero times it."""
    a, w, _, _ = operands(M, N, K_, M)
    w[w == 0] = 0.1
    want = torch.zeros(M, N, dtype=torch.float64)
    for m, at in enumerate((K_ - 1, 0, K_ - 8, K_ // 2 + 1, K_ // 2 - 130)):
        if m < M:
            a[m, at] = float("inf")
            want[m] = w[:, at].double().sign() * float("inf")
    d_a, d_w = a.to(DEV), w.to(DEV)
    out = torch.zeros(M, N, device=DEV)
    if ranges == 1:
        K.gemm_skinny(out, d_a, d_w, None, K.EPI_F32)
    else:
        K.gemm_skinny(out, d_a, d_w, None, K.EPI_RESIDUAL, ranges, following=(torch.empty(M, N, dtype=torch.bfloat16, device=DEV), torch.ones(N, device=DEV),
                                                                              torch.empty(M, K.fine_stat_tiles(N, M), device=DEV)))
    assert torch.equal(out.cpu().double()[: min(M, 5)], want[: min(M, 5)]) and bool(out[5:].isfinite().all())
