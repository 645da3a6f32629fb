"""Steps of single tokens through the gated delta rule, gated linear attention (recurrent_tokens.hip) and the matrix memory
(matrix_memory.hip) in one launch against the separate kernels, which take a step with an empty run beside them: the same bits in the read-outs, the states and the convolution's inputs.  Widths
at the edges of lanes, columns and wavefronts; one to three value heads a key head; no, few and many taps; runs of two tokens beside empty ones."""

import pytest
import torch

from paged_attention_engine_amd.kernels import lib as K

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
RUNS = [[1], [1, 1, 1, 1, 1], [2, 0, 1], [0, 3, 0]]


def runs_of(lengths, spare):
    """Runs and slots of the sequences; `spare`: an empty run in a slot of its own behind them."""
    rows, at = [], 0
    for n in lengths + ([0] if spare else []):
        rows.append([at, n, 0, 0])
        at += n
    slots = [2 * i + 1 for i in range(len(rows))]
    return torch.tensor(rows, dtype=torch.int32, device=DEV), torch.tensor(slots, dtype=torch.int32, device=DEV)


def normal(gen, *shape):
    return torch.randn(*shape, generator=gen).to(DEV)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("channel", [False, True])
@pytest.mark.parametrize("G,H,D,V,taps", [(1, 1, 36, 1, 1), (2, 4, 64, 256, 4), (6, 12, 128, 128, 4), (2, 6, 100, 72, 7), (3, 3, 68, 65, 2), (1, 2, 40, 200, 5), (2, 8, 64, 40, 3), (1, 5, 36, 16, 4)])
def test_delta_rule(dtype, channel, G, H, D, V, taps):
    gen = torch.Generator().manual_seed(D + V)
    C = 2 * G * D + H * V
    for lengths in RUNS:
        T, S = sum(lengths), len(lengths)
        assert T == S
        proj, gate = normal(gen, T, C + 8).to(dtype), normal(gen, T, H * V + 8).to(dtype)[:, :H * V]
        beta, decay = normal(gen, T, H).to(dtype), normal(gen, T, H * D if channel else H).to(dtype)
        conv_w, a_log, dt = normal(gen, C, taps) * 0.5, normal(gen, H) * 0.3, normal(gen, H * D if channel else H)
        tail, state, norm_w = normal(gen, 2 * S + 4, taps - 1, C), normal(gen, 2 * S + 4, H, V, D), normal(gen, V)
        got = []
        for spare in (False, True):
            runs, slots = runs_of(lengths, spare)
            seq = torch.tensor([s for s, n in enumerate(lengths) for _ in range(n)], dtype=torch.int32, device=DEV)
            out, t, st = torch.full((T, H * V), float("nan"), dtype=dtype, device=DEV), tail.clone(), state.clone()
            K.delta_rule_step(proj, out, seq, torch.zeros_like(seq), runs, slots, conv_w, t, st, a_log, dt, norm_w, G, H, D, V, taps,
                              1e-6, 1e-5, gate=gate, beta=beta, decay_in=decay, channel_decay=channel, gate_activation="sigmoid" if channel else "silu")
            got.append((out, t, st))
        for one, many in zip(*got):
            assert torch.equal(one, many), lengths
        assert not torch.equal(got[0][2], state) and bool(torch.isfinite(got[0][0].float()).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("H,D,V", [(1, 36, 1), (4, 64, 256), (12, 128, 128), (3, 100, 72), (2, 68, 65)])
def test_linear_attention(dtype, bias, H, D, V):
    gen = torch.Generator().manual_seed(D + V)
    for lengths in RUNS:
        T, S = sum(lengths), len(lengths)
        proj, gate = normal(gen, T, 2 * H * D + H * V + 8).to(dtype), normal(gen, T, H * V).to(dtype)
        decay, state, norm_w = normal(gen, T, H * D).to(dtype), normal(gen, 2 * S + 4, H, V, D), normal(gen, V).to(dtype)
        decay_bias = normal(gen, H * D) if bias else None
        got = []
        for spare in (False, True):
            runs, slots = runs_of(lengths, spare)
            out, st = torch.full((T, H * V), float("nan"), dtype=dtype, device=DEV), state.clone()
            K.linear_attention_step(proj, decay, decay_bias, 16.0, gate, out, runs, slots, st, norm_w, H, D, V, 1e-5, "silu" if bias else "sigmoid")
            got.append((out, st))
        for one, many in zip(*got):
            assert torch.equal(one, many), lengths
        assert not torch.equal(got[0][1], state) and bool(torch.isfinite(got[0][0].float()).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("formed", [False, True])
@pytest.mark.parametrize("H,D,V,hidden", [(1, 4, 1, 64), (4, 64, 128, 1536), (12, 128, 128, 1536), (3, 100, 72, 100), (2, 68, 65, 1030)])
def test_matrix_memory(dtype, formed, H, D, V, hidden):
    gen = torch.Generator().manual_seed(D + V)
    for lengths in RUNS:
        T, S = sum(lengths), len(lengths)
        proj, gate = normal(gen, T, 2 * H * D + H * V).to(dtype), normal(gen, T, H * V).to(dtype)
        x, gate_w, gate_b = normal(gen, T, hidden).to(dtype), (normal(gen, 2 * H, hidden) * 0.1).to(dtype), normal(gen, 2 * H) * 3.0
        logits = None if formed else normal(gen, T, 2 * H) * 6.0
        state, maximum, norm_w = normal(gen, 2 * S + 4, H, V + 1, D), normal(gen, 2 * S + 4, H), normal(gen, H * V)
        empty, got = torch.zeros(0, 4, dtype=torch.int32, device=DEV), []
        for spare in (False, True):
            runs, slots = runs_of(lengths, spare)
            serial = torch.stack([torch.arange(len(runs), dtype=torch.int32, device=DEV), runs[:, 0], runs[:, 1], runs[:, 2]], 1).contiguous()
            out, st, top = torch.full((T, H * V), float("nan"), dtype=dtype, device=DEV), state.clone(), maximum.clone()
            K.matrix_memory_step(proj, gate, logits, out, serial, empty, empty, slots, st, top, norm_w, H, D, V, 15.0, 1e-5, 1e-6,
                                 gates_from=(x, gate_w, gate_b) if formed else None)
            got.append((out, st, top))
        for one, many in zip(*got):
            assert torch.equal(one, many), lengths
        assert not torch.equal(got[0][1], state) and bool(torch.isfinite(got[0][0].float()).all())
