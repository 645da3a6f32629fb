"""Products of many rows (csrc/gemm_wide.hip) against the same in 64 bits, over every tile shape: edges and remainders of
tiles in rows and features, the fewest stages of k, what is left over behind whole rounds of tiles in halves and quarters, operands that are
rows of wider ones.  A sum's order depends on k alone, so every shape gives the same bits."""

import pytest
import torch

from paged_attention_engine_amd.kernels import lib as K

pytestmark = pytest.mark.gpu

SHAPES = range(6)
GATED_SHAPES = (0, 1, 2, 4, 5)
SUMS_SHAPES = (1, 2, 3, 4, 5)
GUARD = 64  # rows behind the result, which must stay as they are

# rows, features, k
SIZES = [(65, 16, 128), (64 + 1, 48, 192), (127, 144, 128), (128, 256, 256), (129, 272, 320), (255, 1168, 128), (257, 528, 448),
         (300, 96, 1536), (513, 1552, 896),
         (513, 21856, 128),   # 3 x 86 tiles of 256 x 256: two left over behind a round, in quarters, and the last of them 96 wide
         (1100, 17920, 128),  # 5 x 70: 94 left over, in halves, rows that end inside a half
         (2048, 17920, 192)]  # 8 x 70: 48 left over, in quarters


def operands(M, N, k, seed=0, wider=0):
    gen = torch.Generator(device="cuda").manual_seed(seed + M + N + k)
    a = torch.randn(M, k + wider, generator=gen, device="cuda").to(torch.bfloat16)[:, :k]
    w = (torch.randn(N, k, generator=gen, device="cuda") * k ** -0.5).to(torch.bfloat16)
    return a, w


def guarded(M, N, dtype, lead=None):
    whole = torch.full(((lead or 1) * M + GUARD, N), 7.0, device="cuda", dtype=dtype)
    out = whole[:(lead or 1) * M]
    return (out.view(lead, M, N) if lead else out), whole[(lead or 1) * M:]


def exact(a, w):
    """The product in 64 bits and a bound of the float32 sums' error: k additions, each within half a place (2^-24) of
    a partial sum, which is at most the sum of magnitudes."""
    ref = a.double() @ w.double().T
    return ref, w.shape[1] * 2.0 ** -24 * (a.double().abs() @ w.double().abs().T)


def check(got, ref, err):
    """`err`: of what is rounded to bfloat16 at the end (half a place of its 8 bits: 2^-8)."""
    rounding = 2.0 ** -8 * (ref.abs() + err) if got.dtype == torch.bfloat16 else 0.0
    off = (got.double() - ref).abs() - (err + rounding) * 1.001
    assert float(off.max()) <= 0.0, float(off.max())


@pytest.mark.parametrize("M,N,k", SIZES)
def test_product(M, N, k):
    a, w = operands(M, N, k)
    ref, err = exact(a, w)
    first = None
    for shape in SHAPES:
        out, behind = guarded(M, N, torch.bfloat16)
        K.gemm_wide(out, a, w, shape | 1 << 8)
        check(out, ref, err)
        assert bool((behind == 7.0).all())
        first = out if first is None else first
        assert torch.equal(out, first), shape


@pytest.mark.parametrize("M,N,k", [(65, 16, 128), (129, 272, 320), (513, 1552, 896), (513, 21856, 128)])
@pytest.mark.parametrize("kind", [None, "gelu", "relu2"])
def test_bias_and_activation(M, N, k, kind):
    a, w = operands(M, N, k, 1, wider=24)
    bias = torch.randn(N, device="cuda")
    for b in (bias, bias.to(torch.bfloat16)):
        ref, err = exact(a, w)
        if kind is not None:  # the activation reads the sum rounded to bfloat16
            err = err + 2.0 ** -8 * (ref.abs() + err)
        ref = ref + b.double()
        err = err + 2.0 ** -24 * (ref.abs() + err)
        if kind == "gelu":  # its slope is at most 1.13; erff and what is around it: a few places
            ref, err = torch.nn.functional.gelu(ref), 1.13 * err + 8 * 2.0 ** -24 * (ref.abs() + 1.0)
        elif kind == "relu2":
            ref, err = torch.relu(ref).pow(2), (2 * ref.abs() + err) * err + 2.0 ** -23 * (ref.abs() + err).pow(2)
        for shape in SHAPES:
            out, behind = guarded(M, N, torch.bfloat16)
            K.gemm_wide(out, a, w, shape | 1 << 8, b, kind)
            check(out, ref, err)
            assert bool((behind == 7.0).all())


@pytest.mark.parametrize("M,N,k", [(65, 16, 128), (129, 272, 320), (257, 528, 448), (513, 21856, 128), (1100, 17920, 128)])
@pytest.mark.parametrize("kind", ["silu", "gelu_tanh"])
def test_gated(M, N, k, kind):
    a, w = operands(M, N, k, 2, wider=8)
    ref, err = exact(a, w)
    err = err + 2.0 ** -8 * (ref.abs() + err)  # both factors are read rounded to bfloat16
    pair, off = ref.view(M, N // 16, 2, 8), err.view(M, N // 16, 2, 8)
    g, u, dg, du = (t.reshape(M, N // 2) for t in (pair[:, :, 0], pair[:, :, 1], off[:, :, 0], off[:, :, 1]))
    act = torch.nn.functional.silu(g) if kind == "silu" else torch.nn.functional.gelu(g, approximate="tanh")
    # both slopes are at most 1.13; expf, tanhf and what is around them: within 2^-20 of the argument's size
    da = 1.13 * dg + 2.0 ** -20 * (g.abs() + 1.0) * (1.0 + dg)
    ref, err = act * u, act.abs() * du + (u.abs() + du) * da + 2.0 ** -24 * (act * u).abs()
    for shape in GATED_SHAPES:
        out, behind = guarded(M, N // 2, torch.bfloat16)
        K.gemm_wide(out, a, w, shape | 1 << 8, kind=kind, mode=K.WIDE_GATED)
        check(out, ref, err)
        assert bool((behind == 7.0).all())


@pytest.mark.parametrize("M,N,k,ranges", [(65, 16, 64, 1), (129, 272, 320, 2), (257, 528, 448, 7), (513, 1552, 896, 3)])
def test_sums_of_ranges(M, N, k, ranges):
    a, w = operands(M, N, k, 3)
    at = [k // 64 * i // ranges * 64 for i in range(ranges + 1)]
    for shape in SUMS_SHAPES:
        out, behind = guarded(M, N, torch.float32, ranges)
        K.gemm_wide(out, a, w, shape | ranges << 8, mode=K.WIDE_SUMS)
        for i in range(ranges):
            check(out[i], *exact(a[:, at[i]:at[i + 1]], w[:, at[i]:at[i + 1]]))
        assert bool((behind == 7.0).all())


@pytest.mark.parametrize("M,N,k,ranges", [(65, 16, 128, 1), (129, 272, 320, 2), (257, 528, 448, 3), (513, 1552, 896, 7), (300, 4112, 1216, 4)])
def test_sums_of_ranges_in_the_largest_tiles(M, N, k, ranges):
    """Two stages a range and more, odd numbers of them, more tiles than one and ranges of unequal length."""
    a, w = operands(M, N, k, 3)
    at = [k // 64 * i // ranges * 64 for i in range(ranges + 1)]
    out, behind = guarded(M, N, torch.float32, ranges)
    K.gemm_wide(out, a, w, ranges << 8, mode=K.WIDE_SUMS)
    for i in range(ranges):
        check(out[i], *exact(a[:, at[i]:at[i + 1]], w[:, at[i]:at[i + 1]]))
    assert bool((behind == 7.0).all())
    with pytest.raises(K.KernelError):  # a range of one stage
        K.gemm_wide(torch.empty((k // 64, M, N), device="cuda"), a, w, k // 64 << 8, mode=K.WIDE_SUMS)


@pytest.mark.parametrize("M,N,k", [(129, 272, 320), (1100, 17920, 128)])
def test_same_bits_as_two_kernels(M, N, k):
    a, w = operands(M, N, k, 5)
    product = torch.empty((M, N), device="cuda", dtype=torch.bfloat16)
    K.gemm_wide(product, a, w, 2 | 1 << 8)
    bias = torch.randn(N, device="cuda")
    for kind in K.WIDE_ACTIVATIONS[K.WIDE_PLAIN]:
        want, got = product.clone(), torch.empty_like(product)
        K.activation(want, kind, bias)
        K.gemm_wide(got, a, w, 0 | 1 << 8, bias, kind)
        assert torch.equal(got, want), kind
    for kind in K.WIDE_ACTIVATIONS[K.WIDE_GATED]:
        want, got = (torch.empty((M, N // 2), device="cuda", dtype=torch.bfloat16) for _ in range(2))
        (K.swiglu if kind == "silu" else lambda o, x, block: K.gated_act(o, x, kind, block))(want, product, 8)
        K.gemm_wide(got, a, w, 0 | 1 << 8, kind=kind, mode=K.WIDE_GATED)
        assert torch.equal(got, want), kind


def test_which_products_are_taken():
    a, w = operands(100, 1536, 1536)
    assert K.wide_plan(a, w) is not None
    plan = K.wide_plan(*operands(100, 1536, 8960), K.WIDE_SUMS, ranges=True)
    assert plan >> 8 > 1  # few tiles and much of k
    for bad in (a[:64], a.float(), a[:, 1:], a.t()):
        assert K.wide_plan(bad, w) is None
    wide = operands(100, 1536, 1544)[0]
    assert K.wide_plan(wide[:, :1536], w) is not None  # rows of a wider matrix
    assert K.wide_plan(wide[:, 4:1540], w) is None     # that begin between two multiples of 16 bytes
    assert K.wide_plan(operands(100, 1536, 96)[0], operands(100, 1536, 96)[1]) is None
    assert K.wide_plan(a, w[:1530]) is None
    assert K.wide_plan(a, w, K.WIDE_GATED, "gelu") is None and K.wide_plan(a, w, K.WIDE_GATED, "silu") is not None


def test_linear_with_odd_operands():
    """Products that the tiles do not take go to the library, with the same meaning."""
    from paged_attention_engine_amd.parts.linear import Linear

    for M, N, k in ((70, 1530, 200), (70, 50, 96), (100, 256, 256)):
        a, w = operands(M, N, k, 4)
        bias = torch.randn(N, device="cuda")
        ref, err = exact(a, w)
        for b in (None, bias):
            want = ref if b is None else ref + b.to(torch.bfloat16).double()
            got = Linear(w, None if b is None else b.to(torch.bfloat16))(a)
            # (the library may round the product before it adds the bias)
            check(got, want, err + 2.0 ** -7 * ref.abs())


def test_linear_with_odd_biases():
    """A bias that does not lie number by number, or is one number for all, goes to the library; shapes that do not fit are refused there."""
    from paged_attention_engine_amd.parts.linear import Linear

    a, w = operands(100, 256, 256, 6)
    wide = torch.randn(2 * 256, device="cuda").to(torch.bfloat16)
    for bias in (wide[::2], wide[:1], wide[:256].to(torch.float16)):
        ref, err = exact(a, w)
        want = ref + bias.to(torch.bfloat16).double()
        check(Linear(w, bias)(a), want, err + 2.0 ** -7 * ref.abs())
    with pytest.raises(RuntimeError):
        Linear(w)(a[:, :128].contiguous())


@pytest.mark.parametrize("M", [65, 130, 300])
@pytest.mark.parametrize("nh,nkv,hd,rot,bs,bias,k", [(12, 2, 128, 128, 16, True, 192), (7, 1, 64, 64, 16, False, 128), (3, 3, 192, 64, 32, True, 128),
                                                     (5, 1, 128, 64, 8, True, 128), (4, 0, 64, 64, 16, True, 128), (2, 2, 64, 0, 16, False, 128)])
def test_projections_rotate_and_store(M, nh, nkv, hd, rot, bs, bias, k):
    """In every tile shape: queries rotated, keys rotated and values in their pages, nothing beside them written."""
    from tests.plain import qwen2_plain as plain

    N = (nh + 2 * nkv) * hd
    gen = torch.Generator().manual_seed(M + N)
    a, w = torch.randn(M, k, generator=gen).bfloat16(), (torch.randn(N, k, generator=gen) * k ** -0.5).bfloat16()
    b = torch.randn(N, generator=gen).bfloat16() if bias else None
    positions = torch.arange(2, 2 + 2 * M, 2, dtype=torch.int32) // 3 * 2  # not one after another
    positions, tok_seq = positions + torch.arange(M, dtype=torch.int32) % 2, torch.arange(M, dtype=torch.int32) % 7
    blocks = int(positions.max()) // bs + 1
    tables = torch.randperm(7 * blocks, generator=gen).int().view(7, blocks)
    x = (a.double() @ w.double().t() + (b.double() if bias else 0.0)).bfloat16().double().view(M, -1, hd)
    turned = x.clone()
    if rot:
        cos, sin = plain.rope_cos_sin(plain.rope_inv_freq(rot, 1e4, torch.float64), positions, torch.float64)
        turned[..., :rot] = x[..., :rot] * cos[:, None] + plain.rotate_half(x[..., :rot]) * sin[:, None]
    dev = lambda t: t.cuda() if t is not None else None
    angles = K.rope_table(positions.cuda(), plain.rope_inv_freq(rot, 1e4).cuda()) if rot else None
    # the projection's rounding may fall the other way (2^-7 of it), of each of a rotated pair, and the result is rounded
    bound = 2.0 ** -7 * (x.abs().amax(-1, keepdim=True) * 1.5 + 0.01)
    assert K.wide_rope_plan(dev(a), dev(w), hd, rot, dev(b)) is not None
    for shape in GATED_SHAPES:
        pools = [torch.full((7 * blocks, nkv, *s), 7.0, dtype=torch.bfloat16, device="cuda") for s in ((bs, hd), (hd, bs))] if nkv else [None, None]
        q = torch.full((M, nh * hd + 8), 7.0, dtype=torch.bfloat16, device="cuda")
        K.gemm_wide_rope(q[:, :nh * hd], dev(a), dev(w), dev(b), shape | 1 << 8, nh, nkv, hd, rot, angles, dev(positions), dev(tok_seq) if nkv else None,
                         dev(tables) if nkv else None, bs, *pools)
        assert ((q[:, :nh * hd].double().cpu().view(M, nh, hd) - turned[:, :nh]).abs() <= bound[:, :nh]).all()
        assert bool((q[:, nh * hd:] == 7.0).all())
        if not nkv:
            continue
        last = {(int(tok_seq[m]), int(positions[m])): m for m in range(M)}  # the rows whose slot no later row takes
        pages, at = [int(tables[s, p // bs]) for s, p in last], [p % bs for _, p in last]
        rows = list(last.values())
        assert len(rows) == M
        assert ((pools[0].cpu().double()[pages, :, at] - turned[rows, nh:nh + nkv]).abs() <= bound[rows, nh:nh + nkv]).all()
        assert ((pools[1].cpu().double()[pages, :, :, at] - x[rows, nh + nkv:]).abs() <= bound[rows, nh + nkv:]).all()
        kept = torch.ones(7 * blocks, bs, dtype=torch.bool)
        kept[pages, at] = False
        assert bool((pools[0].cpu().transpose(1, 2)[kept] == 7.0).all()) and bool((pools[1].cpu().permute(0, 3, 1, 2)[kept] == 7.0).all())


@pytest.mark.parametrize("kind", ["silu", "gelu_tanh", "gelu"])
def test_activations_of_every_bfloat16_number(kind):
    """Activations of bfloat16 results are worked out by the unit's own exponential and reciprocal: within bfloat16's rounding, 2^-8 of the
    result and a part in 100 more, of the activation in float64.  Left out is what the unit gives as zero: results below 3e-37, from where
    exp(-z) passes float32's largest number (-88.72) or exp(-z^2 / 2) its least.  What is not finite stays so."""
    z = torch.arange(65536, dtype=torch.int32).to(torch.int16).view(torch.bfloat16)
    x = torch.zeros(1, 2 * 65536, dtype=torch.bfloat16)
    x[0, :65536], x[0, 65536:] = z, 1.0
    x, d = x.to("cuda"), z.double()
    if kind == "gelu":
        exact = 0.5 * d * torch.special.erfc(-d * 0.5 ** 0.5)
    else:
        exact = d / (1 + torch.exp(-d if kind == "silu" else -2 * (2 / torch.pi) ** 0.5 * (d + 0.044715 * d ** 3)))
    finite = z.isfinite()
    calls = [lambda out: K.gated_act(out, x, kind)]
    calls += {"silu": [lambda out: K.swiglu(out, x)], "gelu": [lambda out: K.activation(out.copy_(x[:, :65536]), kind)], "gelu_tanh": []}[kind]
    for call in calls:
        out = torch.empty(1, 65536, dtype=torch.bfloat16, device="cuda")
        call(out)
        got = out[0].cpu().double()
        assert ((got - exact).abs() <= 2.0 ** -8 * 1.01 * exact.abs() + 2.0 ** -133 + 3e-37 * (exact.abs() < 3e-37))[finite].all()
        assert torch.equal(got.isnan(), exact.isnan()) and got[z == float("inf")] == float("inf")


def run_whole(M, N, ranges=1):
    """How many tiles of 256 x 256 are run as such: what is left over behind whole rounds of 256 is cut where it is half a round or less."""
    tiles = -(-M // 256) * -(-N // 256)
    return tiles * ranges if ranges > 1 or tiles % 256 > 128 else tiles - tiles % 256


@pytest.mark.parametrize("M,N,mode,ranges,kind", [
    (4097, 8208, K.WIDE_PLAIN, 1, None), (2048, 17920, K.WIDE_GATED, 1, "silu"), (2300, 11504, K.WIDE_GATED, 1, "silu"),
    (2300, 11504, K.WIDE_GATED, 1, "gelu_tanh"), (2300, 11504, K.WIDE_PLAIN, 1, "gelu"), (2100, 11504, K.WIDE_PLAIN, 1, None), (1000, 9216, K.WIDE_SUMS, 4, None)])
def test_more_tiles_of_256_than_units(M, N, mode, ranges, kind):
    """A workgroup then takes one tile after another: what its first tile gives and its last, with whole tiles, cut ones and ranges of k,
    is what tiles of 128 x 128 give, bit for bit; all workgroups two (2,048 rows, gated), or some of them."""
    a, w = operands(M, N, 512, 9)
    bias = torch.randn(N, device="cuda") if mode == K.WIDE_PLAIN else None
    shape = {K.WIDE_PLAIN: (M, N), K.WIDE_GATED: (M, N // 2), K.WIDE_SUMS: (ranges, M, N)}[mode]
    got = [torch.full(shape, float("nan"), device="cuda", dtype=torch.float32 if mode == K.WIDE_SUMS else torch.bfloat16) for _ in range(2)]
    for out, tile in zip(got, (0, 2)):
        K.gemm_wide(out, a, w, tile | ranges << 8, bias, kind=kind, mode=mode)
    assert run_whole(M, N, ranges) > 256 and torch.equal(*got)


def test_more_tiles_of_256_than_units_of_heads():
    """A workgroup a tile here; queries, keys and values are those of tiles of 128 x 128."""
    M, nh, nkv, hd, bs = 5408, 28, 4, 128, 16
    a, w = operands(M, (nh + 2 * nkv) * hd, 256, 3)
    assert run_whole(M, (nh + 2 * nkv) * hd) > 256
    positions, tok_seq = torch.arange(M, device="cuda", dtype=torch.int32), torch.zeros(M, device="cuda", dtype=torch.int32)
    tables = torch.randperm(M // bs, device="cuda").int()[None].contiguous()
    angles = torch.randn(M, hd // 2, 2, device="cuda")
    got = []
    for tile in (0, 2):
        q = torch.empty(M, nh * hd, device="cuda", dtype=torch.bfloat16)
        pools = [torch.empty(M // bs, nkv, *s, device="cuda", dtype=torch.bfloat16) for s in ((bs, hd), (hd, bs))]
        K.gemm_wide_rope(q, a, w, None, tile | 1 << 8, nh, nkv, hd, hd, angles, positions, tok_seq, tables, bs, *pools)
        got.append((q, *pools))
    assert all(torch.equal(x, y) for x, y in zip(*got)) and bool(got[0][1].float().isfinite().all())


@pytest.mark.parametrize("kind,low,bound", [("silu", -88.0, 3e-7), ("gelu_tanh", -1.0, 3.5e-7), ("gelu", -1.0, 4.5e-7)])
def test_gates_round_once(kind, low, bound):
    """act(g) u is worked out in float32 and rounded: no result lies farther from the product in float64 than half a place of bfloat16 and the error of
    float32, which is measured here, over some 2,000 g by all 128 mantissas of u, by the results next to a tie.  The bounds are twice what act_of (1.7e-7
    for SiLU, 2.3e-7 and 3.3e-7 for GELU above -1, where 1 + tanh and 1 + erf are not yet small) and the product's own rounding (6e-8) come to at most,
    and below what an exponential of a rounded product leaves (5e-7 at -8, 4e-6 at -88)."""
    g = torch.arange(65536, dtype=torch.int32).to(torch.int16).view(torch.bfloat16)
    g = g[(g.abs().float() >= 2.0 ** -10) & (g.float() >= low) & (g.float() <= 88.0)]
    u = (1 + torch.arange(128) / 128).to(torch.bfloat16)
    x = torch.cat([g[None].expand(128, -1), u[:, None].expand(-1, len(g))], 1).contiguous()
    d = g.double()
    if kind == "gelu":
        act = 0.5 * d * torch.special.erfc(-d * 0.5 ** 0.5)
    else:
        act = d / (1 + torch.exp(-d if kind == "silu" else -2 * (2 / torch.pi) ** 0.5 * (d + 0.044715 * d ** 3)))
    exact = act[None] * u.double()[:, None]
    half_place = 2.0 ** (torch.frexp(exact)[1].double() - 9)
    calls = [lambda out: K.gated_act(out, x.to("cuda"), kind)] + ([lambda out: K.swiglu(out, x.to("cuda"))] if kind == "silu" else [])
    for call in calls:
        out = torch.empty(exact.shape, dtype=torch.bfloat16, device="cuda")
        call(out)
        beyond = ((out.cpu().double() - exact).abs() - half_place) / exact.abs()
        assert float(beyond.max()) <= bound
