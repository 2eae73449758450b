"""The gated delta rule 64 tokens at a time, and of a step of single tokens in one launch (``csrc/gated_delta.hip``),
against its recurrence in 64 bits, beside the token-by-token kernel on the same inputs."""
import types

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
EPS, FLOOR = 1e-5, 1e-6

CASES = [  # (segment lengths, H, G, dk, dv, what is special)
    ([64], 2, 2, 128, 128, ""),                            # one whole chunk
    ([1, 65, 3, 200, 31, 32], 4, 2, 128, 48, ""),          # one token over, short segments between, a chunk of 8
    ([129, 63], 3, 1, 64, 16, ""),                         # the other key size, one tile of values
    ([300], 2, 1, 128, 256, "strong decays"),              # products of decays underflow within a chunk, weak ones after
    ([257], 2, 2, 128, 128, "one key again and again"),    # L is full: every token writes over what the last one wrote
    ([1] * 5, 4, 2, 128, 128, ""),                         # single tokens
    ([1], 3, 3, 64, 40, ""),                               # values that fill no turn of the block's columns
    ([1] * 3, 2, 1, 64, 256, "strong decays"),
]


def recurrence(rows, gates, a_log, dt_bias, S, H, G, dk, dv):
    q, k, v = rows.double().split([G * dk, G * dk, H * dv], 1)
    unit = lambda x: x / torch.sqrt((x * x).sum(-1, keepdim=True) + FLOOR)
    q, k = (unit(x.reshape(-1, G, dk)).repeat_interleave(H // G, 1) for x in (q, k))
    q, v = q * dk ** -0.5, v.reshape(-1, H, dv)
    beta = torch.sigmoid(gates[:, :H].double())
    decay = torch.exp(-torch.exp(a_log.double()) * torch.nn.functional.softplus(gates[:, H:].double() + dt_bias.double()))
    S, out = S.double().transpose(1, 2).clone(), []  # [H, dk, dv]
    for t in range(rows.shape[0]):
        S = decay[t][:, None, None] * S
        u = beta[t][:, None] * (v[t] - (k[t][:, None] @ S)[:, 0])
        S = S + k[t][:, :, None] * u[:, None]
        out.append((q[t][:, None] @ S)[:, 0])
    return torch.stack(out), S.transpose(1, 2)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("lens, H, G, dk, dv, special", CASES)
def test_chunks_against_the_recurrence(lens, H, G, dk, dv, special, dtype):
    from jax_llm_examples_amd.engine import get_ops
    ops = get_ops(DEV)
    g = torch.Generator().manual_seed(sum(lens) + dk + dv)
    N, R = sum(lens), len(lens)
    rn = lambda *s: torch.randn(*s, generator=g)
    rows, gates = rn(N, 2 * G * dk + H * dv).to(dtype), rn(N, 2 * H)
    a_log, dt_bias = rn(H) - 1.0, rn(H)
    if special == "strong decays":
        a_log = torch.full((H,), 3.0)
        gates[:, H:] = torch.where(torch.rand(N, H, generator=g) < 0.1, 6.0, -6.0)
    if special == "one key again and again":
        rows[:, G * dk: 2 * G * dk] = rows[0, G * dk: 2 * G * dk] + 0.01 * rows[:, G * dk: 2 * G * dk]
        gates[:, :H] = 4.0
        a_log[:] = -8.0
    norm, gate = torch.rand(dv, generator=g) + 0.5, rn(N, H * dv).to(dtype)
    slots, phase = torch.randperm(R + 1, generator=g)[:R].int(), torch.tensor([i % 2 for i in range(R)], dtype=torch.int32)
    state = rn(R + 1, 2, H, dv, dk)
    cu = torch.tensor([0] + lens).cumsum(0).int()
    got = {}
    for way, first in (("chunks", 32), ("scan", 1 << 30)):  # ("chunks": or, of single tokens, the one launch)
        ops.DELTA_CHUNKS_FROM, ops.DELTA_CHUNKS_LONG = first, 1
        ctx = types.SimpleNamespace(seg_lens=lens, num_segments=R, cu_seqlens=cu.to(DEV), state_slots=slots.to(DEV),
                                    state_phase=phase.to(DEV), scratch={},
                                    max_seg_len=max(lens) if way == "chunks" else 2)
        st = state.to(DEV)
        o = ops.gated_delta(rows.to(DEV), gates.to(DEV), a_log.to(DEV), dt_bias.to(DEV), norm.to(DEV), gate.to(DEV), H, G,
                            dk, dv, EPS, FLOOR, st, ctx)
        got[way] = o.cpu().double(), st.cpu().double()
    want, want_state = [], state.double().clone()
    for i in range(R):
        part = slice(int(cu[i]), int(cu[i + 1]))
        o, S = recurrence(rows[part], gates[part], a_log, dt_bias, state[slots[i], phase[i]], H, G, dk, dv)
        want.append(o)
        want_state[slots[i], 1 - phase[i]] = S
    o = torch.cat(want)
    o = o / torch.sqrt((o * o).mean(-1, keepdim=True) + EPS) * norm.double()
    z = gate.double()
    o = o.flatten(1) * z * torch.sigmoid(z)
    err = {way: [float((a - b).norm() / b.norm()) for a, b in zip(v, (o, want_state))] for way, v in got.items()}
    # float32 sums of some hundred terms in another order; the result rounded to bfloat16 where that is the run dtype
    for a, b in zip(err["chunks"], err["scan"]):
        assert a < 2 * b + 2e-7, err
    assert err["chunks"][1] < 2e-6 and err["chunks"][0] < (2e-6 if dtype == torch.float32 else 3e-3), err


@pytest.mark.parametrize("where", ["value", "key", "query", "write strength", "decay", "memory"])
@pytest.mark.parametrize("what", [float("nan"), float("inf"), -float("inf")])
def test_what_is_not_finite_reaches_no_token_before_it(where, what):
    """An infinity or NaN within a chunk gives what the recurrence token by token gives: the tokens before it, other heads
    and other columns of the memory keep their numbers."""
    from jax_llm_examples_amd.engine import get_ops
    ops = get_ops(DEV)
    lens, H, G, dk, dv, bad = [150, 70], 2, 1, 128, 48, 100  # (in the first segment's second chunk)
    g = torch.Generator().manual_seed(5)
    N, R = sum(lens), len(lens)
    rn = lambda *s: torch.randn(*s, generator=g)
    rows, gates, state = rn(N, 2 * G * dk + H * dv), rn(N, 2 * H), rn(R, 2, H, dv, dk)
    a_log, dt_bias, norm, gate = rn(H) - 1.0, rn(H), torch.rand(dv, generator=g) + 0.5, rn(N, H * dv)
    if where == "memory":
        state[0, 0, 1, 17, 5] = what
    elif where in ("write strength", "decay"):
        gates[bad, {"write strength": 0, "decay": H}[where] + 1] = what
    else:
        rows[bad, {"query": 3, "key": G * dk + 3, "value": 2 * G * dk + dv + 20}[where]] = what
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)
    got = {}
    for way, first in (("chunks", 32), ("scan", 1 << 30)):
        ops.DELTA_CHUNKS_FROM, ops.DELTA_CHUNKS_LONG = first, 1
        ctx = types.SimpleNamespace(seg_lens=lens, num_segments=R, cu_seqlens=i32([0, 150, 220]), state_slots=i32([0, 1]),
                                    state_phase=i32([0, 1]), scratch={}, max_seg_len=max(lens))
        st = state.to(DEV)
        o = ops.gated_delta(*(x.to(DEV) for x in (rows, gates, a_log, dt_bias, norm, gate)), H, G, dk, dv, EPS, FLOOR, st, ctx)
        got[way] = o.cpu(), st.cpu()
    for a, b in zip(got["chunks"], got["scan"]):
        for test in (torch.isnan, torch.isposinf, torch.isneginf):
            assert torch.equal(test(a), test(b)), (where, what, int((test(a) != test(b)).sum()))
        f = torch.isfinite(b)
        assert float((a[f] - b[f]).norm() / b[f].norm()) < 2e-6  # (the same sums of float32 numbers in another order)
    if where != "memory":
        assert bool(torch.isfinite(got["chunks"][0][:bad]).all())


@pytest.mark.parametrize("lens", [[100, 40], [1, 1, 1]])
def test_a_memory_that_lies_off_its_16_bytes(lens):
    """Goes token by token, as any memory did before there were chunks."""
    from jax_llm_examples_amd.engine import get_ops
    ops = get_ops(DEV)
    ops.DELTA_CHUNKS_FROM, ops.DELTA_CHUNKS_LONG = 32, 1
    H, G, dk, dv, R, N = 2, 1, 64, 32, len(lens), sum(lens)
    g = torch.Generator(device=DEV).manual_seed(3)
    rn = lambda *s: torch.randn(*s, generator=g, device=DEV)
    args = [rn(N, 2 * G * dk + H * dv), rn(N, 2 * H), rn(H) - 1.0, rn(H), rn(dv), rn(N, H * dv)]
    state = rn(R, 2, H, dv, dk)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)
    got = []
    for off in (0, 1):
        ctx = types.SimpleNamespace(seg_lens=lens, num_segments=R, cu_seqlens=i32([0] + torch.tensor(lens).cumsum(0).tolist()),
                                    state_slots=i32(list(range(R))), state_phase=i32([0] * R), scratch={}, max_seg_len=max(lens))
        st = torch.empty(state.numel() + off, device=DEV)[off:].view(state.shape)
        st.copy_(state)
        o = ops.gated_delta(*args, H, G, dk, dv, EPS, FLOOR, st, ctx)
        got.append((o, st))
    for a, b in zip(*got):
        assert float((a - b).norm() / b.norm()) < 2e-6  # (sums of float32 numbers in two orders)
