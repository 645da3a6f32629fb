"""Prefill attention with keys and values shared through LDS against the formula in 64 bits: at the edges of its groups of 32
tokens, its pages of 16 and tiles of 32 and 64 keys, behind cached tokens, under windows whose earlier pages were given
back, in chunks, with a score cap, sinks, a bias by distance and gates."""

import math

import pytest
import torch

from paged_attention_engine_amd.kernels import lib as K

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def inputs(runs, nh, nkv, hd, vd, seed, gone):
    """Paged keys and values of `runs` [(cached tokens, new tokens)]; pages below `gone[i]` of sequence i are not there, and
    pool page 0, which nobody holds, is full of numbers that are none."""
    gen = torch.Generator().manual_seed(seed)
    randn = lambda *shape: torch.randn(shape, generator=gen).bfloat16()
    pages = [-(-(p + n) // 16) for p, n in runs]
    order = (torch.randperm(sum(pages), generator=gen) + 1).tolist()
    k, v = randn(sum(pages) + 1, nkv, 16, hd), randn(sum(pages) + 1, nkv, vd, 16)
    k[0], v[0] = math.nan, math.inf
    table, keys, values = torch.full((len(runs), max(pages) + 1), -1, dtype=torch.int32), [], []
    for i, (count, (p, n)) in enumerate(zip(pages, runs)):
        mine = [order.pop() for _ in range(count)]
        table[i, :count] = torch.tensor(mine)
        keys.append(k[mine].permute(1, 0, 2, 3).reshape(nkv, -1, hd)[:, :p + n].double())
        values.append(v[mine].permute(1, 0, 3, 2).reshape(nkv, -1, vd)[:, :p + n].double())
        for j in mine[:gone[i]]:
            k[j], v[j] = math.nan, math.inf
        table[i, :gone[i]] = -1
    return randn(sum(n for _, n in runs), nh * hd), k, v, table, keys, values


def exact(q, keys, values, runs, nh, hd, scale, window=0, chunked=False, cap=0.0, sinks=None, slopes=None):
    """The heads [T, nh, vd], and the sums of the weights times the values' sizes."""
    out, sizes, at = [], [], 0
    for (p, n), k, v in zip(runs, keys, values):
        per = nh // k.shape[0]
        s = q[at:at + n].view(n, nh, hd).double().transpose(0, 1) @ k.repeat_interleave(per, 0).transpose(1, 2) * scale
        s = cap * torch.tanh(s / cap) if cap else s
        i, j = torch.arange(p, p + n)[:, None], torch.arange(p + n)[None]
        s = s - slopes.double()[:, None, None] * (i - j) if slopes is not None else s
        hidden = j > i
        if window:
            hidden = hidden | (i // window != j // window if chunked else i - j >= window)
        s = s.masked_fill(hidden, -math.inf)
        if sinks is not None:
            s = torch.cat([s, sinks.double()[:, None, None].expand(-1, n, 1)], -1)
        w = torch.softmax(s, -1)[..., :p + n]
        out.append((w @ v.repeat_interleave(per, 0)).transpose(0, 1))
        sizes.append((w @ v.abs().repeat_interleave(per, 0)).transpose(0, 1))
        at += n
    return torch.cat(out), torch.cat(sizes)


RUNS = {"edges": [(0, 1 + n) for n in (1, 14, 15, 16, 30, 31, 32, 62, 63, 64, 126, 127, 128)], "long": [(0, 700), (0, 257)],
        "behind": [(5, 33), (16, 128), (63, 65), (100, 200), (511, 2), (64, 64)]}
KINDS = {"plain": {}, "window": dict(window=50), "wide window": dict(window=300), "chunks": dict(window=96, chunked=True),
         "cap and sinks": dict(cap=20.0, sinks=True), "distance": dict(slopes=True, gate=True), "head gate": dict(head_gate=True)}


def cases():
    for hd, vd, routes in ((128, 128, (2, 4)), (64, 64, (2,)), (192, 128, (2, 4))):
        for route in routes:
            for kind in KINDS if hd == vd else ("plain", "window", "head gate"):
                for runs in RUNS:
                    yield pytest.param(hd, vd, route, kind, runs, id=f"{hd}-{vd}-{route}-{kind}-{runs}")


@pytest.mark.parametrize("hd,vd,route,kind,runs", cases())
def test_prefill_by_shared_keys(hd, vd, route, kind, runs):
    nh, nkv, scale = 6, 2, hd ** -0.5
    what, runs = dict(KINDS[kind]), RUNS[runs]
    window, chunked, cap = what.get("window", 0), what.get("chunked", False), what.get("cap", 0.0)
    first = lambda p: 0 if not window else p // window * window if chunked else max(0, p - window + 1)
    gone = [first(p) // 16 for p, _ in runs]
    q, k, v, table, keys, values = inputs(runs, nh, nkv, hd, vd, hd + route, gone)
    gen = torch.Generator().manual_seed(1)
    sinks = torch.randn(nh, generator=gen) if "sinks" in what else None
    slopes = 0.2 * torch.rand(nh, generator=gen) if "slopes" in what else None
    gate = torch.randn(len(q), nh * vd, generator=gen).bfloat16() if "gate" in what else None
    head_gate = torch.randn(len(q), nh + 2, generator=gen).bfloat16() if "head_gate" in what else None
    want, sizes = exact(q, keys, values, runs, nh, hd, scale, window, chunked, cap, sinks, slopes)
    tiles, at = [], 0
    for row, (p, n) in enumerate(runs):
        tiles += [(row, at + f, min(K.PREFILL_TILE, n - f)) for f in range(0, n, K.PREFILL_TILE)]
        at += n
    positions = torch.tensor([p + i for p, n in runs for i in range(n)], dtype=torch.int32)
    d = lambda x: x.to(DEV) if x is not None else None
    out = torch.full((len(q), nh * vd + 8), math.nan, dtype=torch.bfloat16, device=DEV)
    qd, kd, vd_, td, pd, bd = (x.to(DEV) for x in (q, k, v, torch.tensor(tiles, dtype=torch.int32), positions, table))
    if hd == vd:
        K.attn_prefill(out[:, :nh * vd], qd, kd, vd_, td, pd, bd, nh, nkv, hd, scale, window, cap, d(sinks), chunked, d(slopes), d(gate),
                       d(head_gate), route=route)
    else:
        hg = d(head_gate)
        assert K.library().pae_attn_prefill_wide_bf16(
            out.data_ptr(), out.stride(0), qd.data_ptr(), qd.stride(0), kd.data_ptr(), vd_.data_ptr(), td.data_ptr(), len(tiles),
            pd.data_ptr(), bd.data_ptr(), bd.shape[1], nh, nkv, hd, vd, scale, window, None, hg.data_ptr() if hg is not None else None,
            hg.stride(0) if hg is not None else 0, len(q), route, torch.cuda.current_stream().cuda_stream) == 0
    got = out[:, :nh * vd].double().cpu().view(-1, nh, vd)
    assert torch.isnan(out[:, nh * vd:]).all()
    # bfloat16 has 8 bits: to the nearest it moves a number by up to 2^-8 of it.  So do the weights (and with them their sum) and the
    # result; scores and sums are float32
    bound = 2.0 ** -8 * (sizes + 2 * want.abs()) + 1e-4
    if gate is not None:
        g = torch.sigmoid(gate.double()).view(-1, nh, vd)
        want, bound = want * g, bound * g
    if head_gate is not None:
        g = torch.sigmoid(head_gate[:, :nh].double())[..., None]
        want, bound = want * g, bound * g
    assert ((got - want).abs() <= bound).all(), float(((got - want).abs() / bound).max())


@pytest.mark.parametrize("R,V,window,pad", [(0, 128, 0, 0), (0, 128, 0, 1), (0, 64, 0, 0), (64, 128, 0, 0), (0, 128, 150, 0)])
def test_formed_heads_with_sinks(R, V, window, pad):
    """Latent attention with the heads formed, with sinks, against 64 bits.  Rows without a rotated part are the queries as they are
    where they start on 16 bytes (`pad` 0)."""
    from paged_attention_engine_amd.parts import StepShape
    from paged_attention_engine_amd.parts.latent import expanded_runs

    gen = torch.Generator().manual_seed(R + V + window)
    H, D, C, bs, runs = 5, 128, 64, 16, [(0, 129), (37, 200)]  # (keys before, new rows)
    bf = lambda x: x.to(torch.bfloat16)
    randn = lambda *shape: torch.randn(*shape, generator=gen)
    w_uk, w_uv, sinks = bf(randn(H * D, C) * C ** -0.5), bf(randn(H * V, C) * C ** -0.5), 3 * randn(H)
    scale, T, past = (D + R) ** -0.5, sum(n for _, n in runs), [a for a, _ in runs]
    width = max(-(-(a + n) // bs) for a, n in runs)
    tables = torch.randperm(2 * width, generator=gen).view(2, width).to(torch.int32)
    pool = bf(randn(2 * width, bs, C + R))
    q = bf(randn(T, H * (D + R) + pad))
    want, sizes, at = [], [], 0
    for s, (a, n) in enumerate(runs):
        rows = pool[tables[s].long()].reshape(-1, C + R)[:a + n].double()
        k = torch.cat([bf(rows[:, :C] @ w_uk.double().T).double().view(-1, H, D), rows[:, None, C:].expand(-1, H, -1)], -1)
        v = bf(rows[:, :C] @ w_uv.double().T).double().view(-1, H, V)
        score = torch.einsum("ihd,jhd->hij", q[at:at + n, :H * (D + R)].double().view(n, H, D + R), k) * scale
        i, j = torch.arange(a, a + n)[:, None], torch.arange(a + n)
        score = score.masked_fill((j > i) | ((i - j >= window) if window else (j < 0)), -math.inf)
        p = torch.softmax(torch.cat([score, sinks.double()[:, None, None].expand(-1, n, 1)], -1), -1)[..., :-1]
        want.append(torch.einsum("hij,jhv->ihv", p, v).reshape(n, -1))
        sizes.append(torch.einsum("hij,jhv->ihv", p, v.abs()).reshape(n, -1))
        at += n
    lists = expanded_runs(StepShape((0, 1), (0, runs[0][1]), tuple(n for _, n in runs), tuple(past), bs), 128, window, K.PREFILL_TILE)
    dev = lambda name: torch.tensor(lists[name][0], dtype=torch.int32, device=DEV).view(-1, lists[name][1])
    positions = torch.cat([torch.arange(a, a + n) for a, n in runs]).to(torch.int32).to(DEV)
    out = torch.full((T, H * V), math.nan, dtype=torch.bfloat16, device=DEV)
    K.latent_expanded(out, q.to(DEV), pool.to(DEV), torch.cat([w_uk, w_uv]).to(DEV), dev("pages"), dev("page_table"), dev("tiles"),
                      positions, tables.to(DEV), None, 1.0, H, D, R, 0, True, V, C, scale, None, window, sinks.to(DEV))
    want, sizes = torch.cat(want), torch.cat(sizes)
    # the roundings of weights, their sum and the result as above; the keys' and values' own, which the oracle repeats, fall on the other
    # side of a tie where the product's sum in 32 bits does: 2^-8 of one of 128 terms of a score, and of a value
    assert ((out.cpu().double() - want).abs() <= 2.0 ** -8 * (2 * sizes + 2 * want.abs()) + 1e-3).all()


def test_runs_choose_a_kernel_by_the_keys_they_see():
    """In tables that a longer sequence made wide: the bits of tables as wide as the run, if the run's keys are told."""
    nh, nkv, hd, n = 12, 2, 128, 100
    q, k, v, table, _, _ = inputs([(0, n)], nh, nkv, hd, hd, 5, [0])
    tiles, at = torch.tensor([[0, 0, n]], dtype=torch.int32, device=DEV), torch.arange(n, dtype=torch.int32, device=DEV)
    wide = torch.full((1, 256), -1, dtype=torch.int32)
    wide[:, :table.shape[1]] = table

    def run(table, **how):
        out = torch.empty(n, nh * hd, dtype=torch.bfloat16, device=DEV)
        K.attn_prefill(out, q.to(DEV), k.to(DEV), v.to(DEV), tiles, at, table.to(DEV), nh, nkv, hd, hd ** -0.5, 0, **how)
        return out

    routes = K.library().pae_attn_prefill_route
    assert routes(nh, hd, hd, 16, 1, n, table.shape[1], 0) == 0 and routes(nh, hd, hd, 16, 1, n, 256, 0) == 2
    assert torch.equal(run(wide, keys=n), run(table)) and torch.equal(run(wide, keys=n), run(wide, route=0))
    assert torch.equal(run(wide), run(wide, route=2))
