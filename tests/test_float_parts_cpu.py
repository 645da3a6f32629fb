"""The three bfloat16 parts of a float32 number (csrc/gemm_plain.hip), taken apart here as the kernels do it: what the six products of parts
leave out of a product, and that a sum without any one of the six is further off than the GPU's tests allow."""

import torch

from tests.test_gpu_kernels import rounded_sums

UPPER = -65536  # the bits of a float32's first half
UP = 65536.0


def parts_of(x):
    """The parts in float64, of the number itself; the kernels hold them times 2^16."""
    bits, number = lambda t: t.contiguous().view(torch.int32), lambda t: t.view(torch.float32)
    x = x * UP
    first = number((bits(x) + 0x8000) & UPPER)
    second = number((bits(x - first) + 0x8000) & UPPER)
    third = x - first - second
    assert torch.equal(number(bits(third) & UPPER), third)
    return [t.double() / UP for t in (first, second, third)]


SIX = [(0, 0), (0, 1), (1, 0), (1, 1), (0, 2), (2, 0)]


def off(a, w, kept):
    """(what `kept` products of parts make of a w) / (a w) - 1"""
    pa, pw, product = parts_of(a), parts_of(w), a.double() * w.double()
    return (sum(pa[i] * pw[j] for i, j in kept) - product) / product


def test_numbers_are_their_parts():
    gen = torch.Generator().manual_seed(1)
    x = torch.randn(100000, generator=gen)
    for scale in (0, 100, -60, -110, -126, -140, -149):
        y = x * 2.0 ** scale if scale > -126 else x * 2.0 ** -100 * 2.0 ** (scale + 100)
        assert torch.equal(sum(parts_of(y)), y.double()), scale


def test_six_products_leave_out_less_than_half_a_unit():
    gen = torch.Generator().manual_seed(2)
    a, w = torch.randn(1000000, generator=gen), torch.randn(1000000, generator=gen)
    hard = torch.tensor([1 + 2.0 ** -8 - 2.0 ** -23, 1 + 2.0 ** -8 - 2.0 ** -17, 1 + 2.0 ** -8 - 2.0 ** -16 - 2.0 ** -17, 2 - 2.0 ** -23])
    a, w = torch.cat([a, hard, -hard, hard]), torch.cat([w, hard, hard, hard.flip(0)])
    err = off(a, w, SIX)
    assert float(err.abs().max()) < 2.0 ** -24
    assert float(err.pow(2).mean().sqrt()) < 2.0 ** -27
    itself = off(a, a, SIX)  # of either sign here too
    assert float(itself.abs().max()) < 2.0 ** -24 and abs(float(itself.mean())) < 2.0 ** -30


def test_a_sum_without_one_of_the_six_is_found():
    gen = torch.Generator().manual_seed(3)
    for k in (32, 1536):
        a, w = torch.randn(20, 1, k, generator=gen), torch.randn(1, 30, k, generator=gen)
        a, w = (t.expand(20, 30, k).reshape(-1) for t in (a, w))
        exact = (a.double() * w.double()).view(600, k)
        for kept in [SIX] + [[p for p in SIX if p != left] for left in SIX]:
            err = (off(a, w, kept).view(600, k) * exact).sum(1).norm() / exact.sum(1).norm()
            assert (float(err) < 0.1 * rounded_sums(k)) if kept is SIX else (float(err) > 1.5 * rounded_sums(k)), (k, kept, float(err))
