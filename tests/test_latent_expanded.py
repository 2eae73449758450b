"""Attention over a cached latent with every head's keys and values formed from it (``csrc/attention_expanded.hip``)
against its definition in 64 bits, and the layout of its work."""
import pytest
import torch

from jax_llm_examples_amd.engine.batch import GroupContext
from jax_llm_examples_amd.ops.hip import HipOps

DN, DR, DV = 128, 64, 128

CASES = [  # (segments: (tokens, position of the first), window, sink, heads, latent, page size)
    ([(130, 0)], None, False, 3, 512, 16),                     # two blocks, the second of two tokens
    ([(64, 0), (129, 0), (127, 5)], None, True, 2, 64, 16),    # a whole step of keys, one token over a block, one short
    ([(33, 700), (200, 64), (96, 63)], None, False, 2, 96, 32),  # tokens cached before, at and beside a step's edge
    ([(257, 1000)], 100, False, 2, 64, 16),                    # a window that begins within a step
    ([(300, 0), (70, 333)], 64, True, 1, 40, 8),               # a window of one step; a latent of odd width
    ([(128, 128)], 1, False, 2, 64, 16),                       # every token sees itself alone
]


@pytest.mark.parametrize("window", [0, 1, 63, 64, 500])
def test_the_plan_covers_every_token_and_every_key_it_sees(window):
    lens, starts = [1, 64, 129, 700, 5], [0, 63, 128, 1000, 777]
    spans, blocks, rows, pairs = HipOps.expanded_plan(lens, starts, window)
    assert len(spans) // 4 * 64 == rows
    assert pairs == sum(min(p + 1, window or p + 1) for n, s in zip(lens, starts) for p in range(s, s + n))
    where = [(i, s + t) for i, (n, s) in enumerate(zip(lens, starts)) for t in range(n)]
    seen = []
    for n0, n, off, _ in (blocks[i: i + 4] for i in range(0, len(blocks), 4)):
        assert 0 < n <= 128
        seg, pos = where[n0]
        assert where[n0: n0 + n] == [(seg, pos + t) for t in range(n)]
        seen += range(n0, n0 + n)
        first = max(0, pos - window + 1) if window else 0
        for kb in range(first // 64 * 64, pos + n, 64):
            span = spans[4 * ((kb + off) // 64):][:4]
            assert (kb + off) % 64 == 0 and span[:2] == [seg, kb] and span[2] <= first and span[3] >= pos + n
    assert sorted(seen) == list(range(len(where)))


@pytest.mark.gpu
@pytest.mark.parametrize("segs, window, sink, H, R, ps", CASES)
def test_against_the_definition(segs, window, sink, H, R, ps):
    dev = "cuda:0"
    ops = HipOps(dev)
    ops.LATENT_EXPAND_PAIRS = 0  # (whatever the sizes)
    g = torch.Generator().manual_seed(len(segs) + R)
    bf = lambda *s, std=1.0: (torch.randn(*s, generator=g) * std).to(torch.bfloat16)
    lens, starts = [n for n, _ in segs], [s for _, s in segs]
    N, width = sum(lens), max(-(-(n + s) // ps) for n, s in segs)
    need = [max(0, s - window + 1) if window else 0 for s in starts]
    table = torch.full((len(segs), width), -1, dtype=torch.int32)
    free = torch.randperm(len(segs) * width, generator=g).tolist()
    for i, (n, s) in enumerate(segs):
        for j in range(need[i] // ps, -(-(n + s) // ps)):  # (pages that no query sees were given back)
            table[i, j] = free.pop()
    latent, rope = bf(len(segs) * width, ps, R), bf(len(segs) * width, ps, DR)
    for i, (n, s) in enumerate(segs):  # what lies behind a segment's end was never written
        if (n + s) % ps:
            latent[table[i, (n + s) // ps], (n + s) % ps:] = float("nan")
            rope[table[i, (n + s) // ps], (n + s) % ps:] = float("nan")
    q = bf(N, H * (DN + DR) + 8)
    uk, uv = bf(H * DN, R, std=R ** -0.5), bf(H * DV, R, std=R ** -0.5)
    sk = torch.randn(H, generator=g) if sink else None
    pos = torch.tensor([s + t for n, s in segs for t in range(n)], dtype=torch.int32)
    seg = torch.tensor([i for i, (n, _) in enumerate(segs) for _ in range(n)], dtype=torch.int32)
    meta = GroupContext(block_table=None, slot_mapping=None, width=width, retention=("all",), seg_lens=lens, seg_starts=starts)
    d = lambda t: None if t is None else t.to(dev)
    scale = (DN + DR) ** -0.5
    got = ops.latent_attention_expanded(d(q)[:, : H * (DN + DR)].view(N, H, DN + DR), DN, d(uk), d(uv), d(latent), d(rope),
                                        d(table), d(pos), d(seg), window, scale, meta, sink=d(sk)).cpu().double()
    o = 0
    for i, (n, s) in enumerate(segs):
        kpos = torch.arange(need[i], s + n)
        c = latent[table[i][kpos // ps].long(), kpos % ps].double()
        kr = rope[table[i][kpos // ps].long(), kpos % ps].double()
        back = torch.arange(s, s + n)[:, None] - kpos[None]
        seen = (back >= 0) & (back < (window or s + n + 1))
        for h in range(H):
            k = torch.cat([c @ uk[h * DN: (h + 1) * DN].double().T, kr], 1)
            qh = q[o: o + n, h * (DN + DR): (h + 1) * (DN + DR)].double()
            sc = (qh @ k.T * scale).masked_fill(~seen, float("-inf"))
            if sink:  # one more key, without a value
                sc = torch.cat([sc, sk[h].double().expand(n, 1)], 1)
            v = c @ uv[h * DV: (h + 1) * DV].double().T
            want = torch.softmax(sc, -1)[:, : len(kpos)] @ v
            err = (got[o: o + n, h * DV: (h + 1) * DV] - want).norm() / want.norm()
            # keys, values, probabilities and the result rounded to bfloat16 (2^-9 each at most, 2^-9 / sqrt(3) rms);
            # a score of size 1 moves by the keys' rounding averaged over 128 terms, far below that
            assert err < 4 * 2.0 ** -9, (i, h, float(err))
        o += n


@pytest.mark.gpu
@pytest.mark.parametrize("window, seen_by", [(None, range(70, 300)), (64, range(70, 134)), (40, range(70, 110))])
@pytest.mark.parametrize("what", [float("nan"), float("inf")])
def test_a_latent_that_is_not_finite_reaches_only_the_tokens_that_see_it(window, seen_by, what):
    """Tokens before its own, and those whose window has passed it, share its steps of 64 keys and keep their numbers."""
    dev, n, H, R, ps = "cuda:0", 300, 2, 64, 16
    ops = HipOps(dev)
    ops.LATENT_EXPAND_PAIRS = 0
    g = torch.Generator().manual_seed(11)
    bf = lambda *s, std=1.0: (torch.randn(*s, generator=g) * std).to(torch.bfloat16).to(dev)
    width = -(-n // ps)
    table = torch.arange(width, dtype=torch.int32, device=dev).view(1, width)
    latent, rope, q = bf(width, ps, R), bf(width, ps, DR), bf(n, H, DN + DR)
    uk, uv = bf(H * DN, R, std=R ** -0.5), bf(H * DV, R, std=R ** -0.5)
    pos, seg = torch.arange(n, dtype=torch.int32, device=dev), torch.zeros(n, dtype=torch.int32, device=dev)
    got = []
    for value in (None, what):
        if value is not None:
            latent[70 // ps, 70 % ps, 5] = value
        meta = GroupContext(block_table=None, slot_mapping=None, width=width, retention=("all",), seg_lens=[n], seg_starts=[0])
        got.append(ops.latent_attention_expanded(q, DN, uk, uv, latent, rope, table, pos, seg, window, (DN + DR) ** -0.5, meta))
    clean, dirty = (x.view(n, H * DV).double() for x in got)
    sees = torch.zeros(n, dtype=torch.bool, device=dev)
    sees[list(seen_by)] = True
    assert not bool(torch.isfinite(dirty[sees]).any())
    # (probabilities not rounded to bfloat16 where a row is formed again, results rounded to it: 2^-9 each)
    assert bool(torch.isfinite(dirty[~sees]).all())
    assert float((dirty - clean)[~sees].norm() / clean[~sees].norm()) < 2.0 ** -8


@pytest.mark.gpu
@pytest.mark.parametrize("first, second", [(2, 8), (8, 2)])
def test_layers_of_unlike_heads_in_one_step_are_judged_by_their_own_sizes(first, second):
    """A step's layout is shared by its layers, what the keys and values take is not: a limit that two heads' keep and
    eight heads' do not."""
    dev, n, R, ps = "cuda:0", 128, 64, 16
    ops = HipOps(dev)
    ops.LATENT_EXPAND_PAIRS = 0
    zeros = lambda *s: torch.zeros(*s, dtype=torch.bfloat16, device=dev)
    table = torch.arange(n // ps, dtype=torch.int32, device=dev).view(1, -1)
    pos, seg = torch.arange(n, dtype=torch.int32, device=dev), torch.zeros(n, dtype=torch.int32, device=dev)
    meta = GroupContext(block_table=None, slot_mapping=None, width=n // ps, retention=("all",), seg_lens=[n], seg_starts=[0])
    taken = lambda H: n * (H * (DN + DV) + R + DR) * 2
    call = lambda H: ops.latent_attention_expanded(zeros(n, H, DN + DR), DN, zeros(H * DN, R), zeros(H * DV, R),
                                                   zeros(n // ps, ps, R), zeros(n // ps, ps, DR), table, pos, seg, None, 0.1, meta)
    ops.LATENT_EXPAND_BYTES = taken(2)
    assert [call(H) is not None for H in (first, second)] == [first == 2, second == 2]
    ops.LATENT_EXPAND_BYTES = taken(2) - 1
    assert call(2) is None


@pytest.mark.gpu
@pytest.mark.parametrize("scale", [0.1, 0.0, -0.1])
def test_every_scale_has_a_way(scale):
    """A scale of zero or below, which a configuration may name, stays in the latent's space."""
    dev, n, H, R, ps = "cuda:0", 80, 2, 64, 16
    ops = HipOps(dev)
    ops.LATENT_EXPAND_PAIRS = 0
    zeros = lambda *s: torch.zeros(*s, dtype=torch.bfloat16, device=dev)
    table = torch.arange(n // ps, dtype=torch.int32, device=dev).view(1, -1)
    pos, seg = torch.arange(n, dtype=torch.int32, device=dev), torch.zeros(n, dtype=torch.int32, device=dev)
    out = ops.latent_attention_expanded(zeros(n, H, DN + DR), DN, zeros(H * DN, R), zeros(H * DV, R), zeros(n // ps, ps, R),
                                        zeros(n // ps, ps, DR), table, pos, seg, None, scale)
    assert (out is not None) == (scale > 0)


@pytest.mark.parametrize("copies", [True, False])
def test_a_mixer_without_the_transposed_latents_keeps_its_float32_probabilities(copies):
    """At widths that the matrix-core kernels do not take (no transposed copies in the cache) attention over the latents is
    float32 arithmetic; keys and values formed once a step are attended to with bfloat16 probabilities."""
    import types
    from jax_llm_examples_amd.parts.latent_attention import LatentAttention
    calls, n = [], 3
    named = lambda name, out=None: lambda *a, **k: (calls.append(name), out)[1]
    ops = types.SimpleNamespace(
        linear=lambda x, w: x @ w.T, batched_linear=lambda x, w, tokens_first=False: torch.zeros(n, 1, DV),
        latent_prepare=named("prepare"), latent_attention=named("latent", torch.zeros(n, 1, 40)),
        latent_attention_expanded=named("expanded", torch.zeros(n, DV)))
    part = types.SimpleNamespace(
        num_heads=1, nope_dim=DN, rope_dim=DR, value_dim=DV, kv_rank=40, own_latent=False, query_rank=None, rotation=None,
        latent_norm_eps=0.0, q_rows=DN + DR, window=None, softmax_scale=1.0, output_gate=False, head_gate=False, w_out=None,
        params={"w_in": torch.zeros(DN + DR, 8), "w_uk": torch.zeros(DN, 40), "w_uv": torch.zeros(DV, 40), "wo": torch.zeros(8, DV)})
    pages = {"latent": None, "rope_key": None, **({"latent_t": None} if copies else {})}
    cache = types.SimpleNamespace(pages=pages, writes=(), block_table=None, slot_mapping=None, attn_meta=None)
    ctx = types.SimpleNamespace(ops=ops, positions=None, token_segment=None)
    assert LatentAttention.forward(part, torch.zeros(n, 8), ctx, cache).shape == (n, 8)
    assert calls == ["prepare", "expanded" if copies else "latent"]


@pytest.mark.gpu
@pytest.mark.parametrize("ps", [4, 8])
def test_pages_that_the_matrix_cores_do_not_take_keep_their_float32_probabilities(ps):
    dev, n, H, R = "cuda:0", 80, 2, 64
    ops = HipOps(dev)
    ops.LATENT_EXPAND_PAIRS = 0
    zeros = lambda *s: torch.zeros(*s, dtype=torch.bfloat16, device=dev)
    table = torch.arange(n // ps, dtype=torch.int32, device=dev).view(1, -1)
    pos, seg = torch.arange(n, dtype=torch.int32, device=dev), torch.zeros(n, dtype=torch.int32, device=dev)
    out = ops.latent_attention_expanded(zeros(n, H, DN + DR), DN, zeros(H * DN, R), zeros(H * DV, R), zeros(n // ps, ps, R),
                                        zeros(n // ps, ps, DR), table, pos, seg, None, 0.1)
    assert (out is not None) == (ps == 8) == bool(ops._query("jle_latent_attention_mfma_supported", R, DN, DR, H * (DN + DR), ps))


@pytest.mark.gpu
@pytest.mark.parametrize("segs, window, sink, H, R, dv, ps", [
    ([(1, 0)], None, False, 1, 32, 4, 8),                                   # one key, the smallest sizes
    ([(1, 126), (1, 127), (1, 128), (1, 159)], None, False, 16, 512, 128, 16),  # beside the edge of a range of 128 keys
    ([(1, 700), (1, 3), (1, 1029)], 128, True, 20, 512, 68, 16),            # windows of one range, tiles of 4 rows, odd widths
    ([(1, 1060 + 50 * i) for i in range(8)], 1024, False, 16, 512, 128, 16),
    ([(5, 100), (1, 31), (17, 64)], 40, False, 3, 160, 64, 32),             # tiles over several tokens, more than 16 tokens
    ([(1, 2000 + i) for i in range(70)], None, True, 16, 256, 96, 16),      # several ranges a block
])
def test_few_rows_through_the_latent_and_out_of_it(segs, window, sink, H, R, dv, ps):
    dev = "cuda:0"
    ops = HipOps(dev)
    g = torch.Generator().manual_seed(len(segs) + R)
    bf = lambda *s, std=1.0: (torch.randn(*s, generator=g) * std).to(torch.bfloat16)
    lens, starts = [n for n, _ in segs], [s for _, s in segs]
    N, width = sum(lens), max(-(-(n + s) // ps) for n, s in segs)
    need = [max(0, s - window + 1) if window else 0 for s in starts]
    table = torch.full((len(segs), width), -1, dtype=torch.int32)
    free = torch.randperm(len(segs) * width, generator=g).tolist()
    latent, rope = bf(len(segs) * width, ps, R), bf(len(segs) * width, ps, DR)
    for i, (n, s) in enumerate(segs):
        for j in range(need[i] // ps, -(-(n + s) // ps)):  # (pages that no query sees were given back)
            table[i, j] = free.pop()
        if (n + s) % ps:  # what lies behind a segment's end was never written
            latent[table[i, (n + s) // ps], (n + s) % ps:] = float("nan")
            rope[table[i, (n + s) // ps], (n + s) % ps:] = float("nan")
    q, q_lat, uv = bf(N, H * (DN + DR) + 8), bf(H, N, R, std=R ** -0.5 * DN ** 0.5), bf(H * dv, R, std=R ** -0.5)
    sk = torch.randn(H, generator=g) if sink else None
    pos = torch.tensor([s + t for n, s in segs for t in range(n)], dtype=torch.int32)
    seg = torch.tensor([i for i, (n, _) in enumerate(segs) for _ in range(n)], dtype=torch.int32)
    single = max(lens) == 1
    meta = GroupContext(block_table=None, slot_mapping=None, width=width, retention=("all",), seg_lens=lens, seg_starts=starts,
                        decode_bucket=-(-max(starts) // 1024) * 1024 + 1024 if single else None)
    d = lambda t: None if t is None else t.to(dev)
    scale = (DN + DR) ** -0.5
    got = ops.latent_values(d(q_lat), d(q)[:, : H * (DN + DR)].view(N, H, DN + DR), DN, d(latent), d(rope), d(table), d(pos),
                            d(seg), window, scale, d(uv), meta=meta, latent_t_pages=d(latent.transpose(1, 2).contiguous()).view(-1, ps, R),
                            sink=d(sk)).cpu().double().view(N, H, dv)
    for t in range(N):
        p, i = int(pos[t]), int(seg[t])
        kpos = torch.arange(max(0, p - window + 1) if window else 0, p + 1)
        c, kr = (x[table[i][kpos // ps].long(), kpos % ps].double() for x in (latent, rope))
        sc = (q_lat[:, t].double() @ c.T + q[t, : H * (DN + DR)].view(H, DN + DR)[:, DN:].double() @ kr.T) * scale
        if sink:
            sc = torch.cat([sc, sk.double()[:, None]], 1)
        out = torch.softmax(sc, -1)[:, : len(kpos)] @ c
        want = torch.einsum("hr,hvr->hv", out, uv.view(H, dv, R).double())
        # probabilities, sums and the result rounded to bfloat16: 2^-9 each at most
        assert (got[t] - want).norm() < 4 * 2.0 ** -9 * want.norm(), (t, float((got[t] - want).norm() / want.norm()))


@pytest.mark.gpu
def test_ranges_whose_scores_are_all_minus_infinity_add_nothing():
    """The first 640 keys' scores overflow to minus infinity: five ranges of 128, as many as the merge takes at a time, have
    no finite maximum before the first that has one."""
    dev, H, R, dv, ps, pos, low = "cuda:0", 16, 64, 32, 16, 1000, 640
    ops = HipOps(dev)
    g = torch.Generator().manual_seed(5)
    bf = lambda *s, std=1.0: (torch.randn(*s, generator=g) * std).to(torch.bfloat16)
    latent, rope = bf(64, ps, R), bf(64, ps, DR)
    q, q_lat, uv = bf(1, H, DN + DR), bf(H, 1, R), bf(H * dv, R, std=R ** -0.5)
    latent[:, :, 0], q_lat[:, :, 0] = 0.0, 1e30
    latent[: low // ps, :, 0] = -1e30
    table, one = torch.arange(64, dtype=torch.int32).view(1, -1), torch.zeros(1, dtype=torch.int32)
    meta = GroupContext(block_table=None, slot_mapping=None, width=64, retention=("all",), seg_lens=[1], seg_starts=[pos],
                        decode_bucket=1024)
    scale = (DN + DR) ** -0.5
    d = lambda t: t.to(dev)
    got = ops.latent_values(d(q_lat), d(q), DN, d(latent), d(rope), d(table), d(one + pos), d(one), None, scale, d(uv), meta=meta,
                            latent_t_pages=d(latent.transpose(1, 2).contiguous()).view(-1, ps, R)).cpu().double().view(H, dv)
    c, kr = latent.view(-1, R)[low: pos + 1].double(), rope.view(-1, DR)[low: pos + 1].double()
    out = torch.softmax((q_lat[:, 0].double() @ c.T + q[0, :, DN:].double() @ kr.T) * scale, -1) @ c
    want = torch.einsum("hr,hvr->hv", out, uv.view(H, dv, R).double())
    # probabilities, sums and the result rounded to bfloat16: 2^-9 each at most
    assert (got - want).norm() < 4 * 2.0 ** -9 * want.norm()
