"""Each HIP kernel alone against its plain PyTorch statement (ops/reference.py), at sizes
other than the engine tests' models: widths and vocabularies that are no power of two,
head sizes in steps of 16, odd head counts and groups."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
DT = [torch.float32, torch.bfloat16]


@pytest.fixture(scope="module")
def ops():
    from jax_llm_examples_amd.engine import get_ops
    return get_ops(DEV)


@pytest.fixture(scope="module")
def ref():
    from jax_llm_examples_amd.ops.reference import ReferenceOps
    return ReferenceOps()


def _tol(dt):
    return dict(rtol=2e-5, atol=2e-6) if dt == torch.float32 else dict(rtol=1.6e-2, atol=1e-3)


def _assert_close_to_scale(got, want, dt):
    """For results that are sums of many rounded terms: error against the size of the whole result."""
    tol = 2e-5 if dt == torch.float32 else 1e-2
    err = float((got.float() - want.float()).abs().max() / want.float().abs().max())
    assert err <= tol, f"error {err:.3g} of the largest value, allowed {tol}"


def _rand(*shape, dt=torch.float32, scale=1.0, seed=None):
    g = torch.Generator(device="cpu").manual_seed(seed if seed is not None else hash(shape) % 1000)
    return (torch.randn(*shape, generator=g) * scale).to(dt).to(DEV)


@pytest.mark.parametrize("dt", DT)
def test_embed(ops, ref, dt):
    table = _rand(311, 80, dt=dt)
    tok = torch.tensor([0, 310, 5, 5, 17], dtype=torch.int32, device=DEV)
    assert torch.equal(ops.embed(tok, table), ref.embed(tok, table))


@pytest.mark.parametrize("dt", DT)
@pytest.mark.parametrize("d", [80, 1000, 1026, 1028, 2056, 5120, 8192, 9000])
def test_add_rmsnorm(ops, ref, dt, d):
    for delta_dt, weighted, want32 in [(None, True, False), (dt, True, True), (torch.float32, False, True)]:
        x = _rand(7, d, seed=1)
        delta = None if delta_dt is None else _rand(7, d, dt=delta_dt, seed=2)
        w = _rand(d, seed=3) if weighted else None
        x1, x2 = x.clone(), x.clone()
        h1, h32_1 = ops.add_rmsnorm(x1, delta, w, 1e-3, dt, want32)
        h2, h32_2 = ref.add_rmsnorm(x2, delta, w, 1e-3, dt, want32)
        assert torch.allclose(x1, x2, rtol=1e-6, atol=1e-6)  # the residual is updated in place, float32
        assert torch.allclose(h1.float(), h2.float(), **_tol(dt))
        if want32:
            assert torch.allclose(h32_1, h32_2, rtol=2e-5, atol=2e-6)
            assert h32_1.dtype == torch.float32


_PIECE_EDGES = [1032, 2048, 2056, 4096, 4104, 6144, 6152, 8192]  # first and last width of two, four, six and eight pieces


@pytest.mark.parametrize("many", [False, True])
@pytest.mark.parametrize("d", _PIECE_EDGES)
def test_add_rmsnorm_at_the_edges_of_its_pieces(ops, d, many):
    """Few rows, and as many as are stored past the caches, against 64 bits."""
    n = -(-(4 << 20) // d) if many else 7
    x, delta, w = _rand(n, d, seed=1), _rand(n, d, dt=torch.bfloat16, seed=2), _rand(d, seed=3)
    want = x.double() + delta.double()
    h, h32 = ops.add_rmsnorm(x, delta, w, 1e-3, torch.bfloat16, True)
    normed = want / torch.sqrt((want ** 2).mean(-1, keepdim=True) + 1e-3) * w.double()
    assert ((x.double() - want).abs() <= 2.0 ** -24 * want.abs()).all()
    # (a thread's up to 32 squares, 8 levels of the sum, root, quotient and products: not 50 roundings of 2^-24)
    assert ((h32.double() - normed).abs() <= 50 * 2.0 ** -24 * normed.abs() + 1e-30).all()
    assert torch.equal(h, h32.bfloat16())


@pytest.mark.parametrize("d", _PIECE_EDGES)
def test_norm_and_router_in_one_launch_at_the_edges_of_its_pieces(ops, d):
    x, delta, w = _rand(5, d, seed=1), _rand(5, d, dt=torch.bfloat16, seed=2), _rand(d, seed=3) + 1.0
    router = _rand(8, d, scale=0.05, seed=4)
    pending = ops.defer_norm(x.clone(), delta, w, 1e-5, torch.bfloat16)
    ids, gates, logits, _ = ops.moe_route(pending, router, 2, want_logits=True, group=True)
    y = x.clone()
    h, h32 = ops.add_rmsnorm(y, delta, w, 1e-5, torch.bfloat16, want32=True)
    assert torch.equal(pending.residual(), y) and torch.equal(pending.rows(), h)
    # (d products of float32 rows, a k of any order, are off by no more than (d + 2) roundings of their sizes' sum)
    want = h32.double() @ router.double().t()
    assert ((logits.double() - want).abs() <= (d + 2) * 2.0 ** -24 * (h32.double().abs() @ router.double().abs().t())).all()
    assert torch.equal(ids.sort(1).values.long(), logits.topk(2, 1).indices.sort(1).values)


def test_rmsnorm_eps_is_inside_the_root(ops):
    x = torch.full((1, 64), 1e-3, device=DEV)
    h, _ = ops.add_rmsnorm(x, None, None, 1e-2, torch.float32)
    assert torch.allclose(h, torch.full_like(h, 1e-3 / math.sqrt(1e-6 + 1e-2)), rtol=1e-5)


@pytest.mark.parametrize("dt", DT)
def test_silu_mul_gather_add(ops, ref, dt):
    for f in (56, 52, 1000):  # halves that are 16-byte aligned (8 elements per thread in bfloat16), and not
        gu = _rand(9, 2 * f, dt=dt, scale=3.0)
        assert torch.allclose(ops.silu_mul(gu).float(), ref.silu_mul(gu).float(), **_tol(dt))
    x = _rand(11, 90, dt=dt)
    idx = torch.tensor([10, 0, 3, 3], dtype=torch.int32, device=DEV)
    assert torch.equal(ops.gather_rows(x, idx), x[idx.long()])
    r, d = _rand(11, 90, seed=4), _rand(11, 90, dt=dt, seed=5)
    want = r + d.float()
    ops.add_residual(r, d)
    assert torch.allclose(r, want, rtol=1e-6, atol=1e-6)


@pytest.mark.parametrize("dt", DT)
def test_qk_prepare_of_a_token_does_not_depend_on_the_batch(ops, ref, dt):
    """Many tokens take wavefronts that go through several heads each; the results must be those of a token
    prepared alone, bit for bit."""
    hq, hk, dh, n, ps = 40, 8, 128, 320, 16
    qkv, pos, pages, slots, inv_freq = _prep_case(hq, hk, dh, n, ps, dt)
    c1 = torch.zeros(pages, 2, hk, ps, dh, dtype=dt, device=DEV)
    c2, c3 = c1.clone(), c1.clone()
    q1 = ops.qk_prepare_kv_write(qkv, hq, hk, dh, pos, _prep(inv_freq, 1e-5, (16.0, 0.1)), c1, slots)
    q2 = ref.qk_prepare_kv_write(qkv, hq, hk, dh, pos, _prep(inv_freq, 1e-5, (16.0, 0.1)), c2, slots)
    assert torch.allclose(q1.float(), q2.float(), **_tol(dt)) and torch.allclose(c1.float(), c2.float(), **_tol(dt))
    few = slice(100, 107)
    q3 = ops.qk_prepare_kv_write(qkv[few].contiguous(), hq, hk, dh, pos[few].contiguous(),
                                 _prep(inv_freq, 1e-5, (16.0, 0.1)), c3, slots[few].contiguous())
    assert torch.equal(q3, q1[few])
    written = c3 != 0
    assert written.any() and torch.equal(c3[written], c1[written])


def _prep(inv_freq=None, eps=None, qs=None, **kw):
    from jax_llm_examples_amd.parts.base import QKPreparation, Rotation

    rot = None if inv_freq is None else Rotation(inv_freq, kw.pop("pairing", "adjacent"), kw.pop("rotary_dim", 0))
    return QKPreparation(rotation=rot, norm_eps=eps, query_scale=qs, **kw)


def _prep_case(hq, hk, dh, n, ps, dt, seed=0):
    qkv = _rand(n, (hq + 2 * hk) * dh, dt=dt, seed=seed)
    pos = torch.randint(0, 500, (n,), generator=torch.Generator().manual_seed(seed)).to(torch.int32).to(DEV)
    pages = 2 * n // ps + 3
    slots = torch.randperm(pages * ps, generator=torch.Generator().manual_seed(seed + 1))[:n].to(torch.int32).to(DEV)
    inv_freq = (1.0 / (10000.0 ** (torch.arange(0, dh, 2).float() / dh))).to(DEV)
    return qkv, pos, pages, slots, inv_freq


@pytest.mark.parametrize("dt", DT)
@pytest.mark.parametrize("hq,hk,dh", [(4, 2, 16), (5, 1, 48), (40, 8, 128), (3, 3, 256), (6, 2, 80)])
def test_qk_prepare_kv_write(ops, ref, dt, hq, hk, dh):
    n, ps = 13, 8
    qkv, pos, pages, slots, inv_freq = _prep_case(hq, hk, dh, n, ps, dt)
    for rope, eps, qs in [(True, 1e-5, None), (False, None, (16.0, 0.1)), (True, None, None), (False, None, None),
                          (True, 1e-3, (4.0, 0.3))]:
        c1 = torch.zeros(pages, 2, hk, ps, dh, dtype=dt, device=DEV)
        c2 = c1.clone()
        q1 = ops.qk_prepare_kv_write(qkv, hq, hk, dh, pos, _prep(inv_freq if rope else None, eps, qs), c1, slots)
        q2 = ref.qk_prepare_kv_write(qkv, hq, hk, dh, pos, _prep(inv_freq if rope else None, eps, qs), c2, slots)
        assert torch.allclose(q1.float(), q2.float(), **_tol(dt))
        assert torch.allclose(c1.float(), c2.float(), **_tol(dt))
        assert (c1[:, 1] != 0).any() and torch.equal(c1 == 0, c2 == 0)  # wrote exactly the same places
    q3 = ops.qk_prepare_kv_write(qkv, hq, hk, dh, pos, _prep(inv_freq), None, None)  # a run that only reads
    assert torch.allclose(q3.float(), ref.qk_prepare_kv_write(qkv, hq, hk, dh, pos, _prep(inv_freq), None,
                                                               None).float(), **_tol(dt))


@pytest.mark.parametrize("dt", DT)
@pytest.mark.parametrize("hq,hk,dh,rd", [(4, 2, 32, 32), (5, 1, 48, 16), (40, 8, 128, 64), (6, 2, 80, 80)])
def test_qk_prepare_other_rotations_and_norms(ops, ref, dt, hq, hk, dh, rd):
    """What Llama 4 does not use but the preparation takes as data: half-split pairs, a rotation of the
    head's leading part only, norm weights, the norm before the rotation."""
    n, ps = 11, 8
    qkv, pos, pages, slots, _ = _prep_case(hq, hk, dh, n, ps, dt, seed=3)
    inv = (1.0 / (10000.0 ** (torch.arange(0, rd, 2).float() / rd))).to(DEV)
    wq, wk = _rand(dh, seed=7) + 1.5, _rand(dh, seed=8) - 1.5
    cases = [dict(pairing="half", rotary_dim=rd), dict(pairing="adjacent", rotary_dim=rd),
             dict(pairing="half", rotary_dim=rd, eps=1e-4, norm_weight_q=wq, norm_weight_k=wk),
             dict(pairing="adjacent", rotary_dim=rd, eps=1e-4, norm_weight_q=wq, norm_weight_k=wk, norm_first=True),
             dict(pairing="half", rotary_dim=rd, eps=1e-2, norm_first=True, qs=(4.0, 0.3))]
    for kw in cases:
        c1 = torch.zeros(pages, 2, hk, ps, dh, dtype=dt, device=DEV)
        c2 = c1.clone()
        q1 = ops.qk_prepare_kv_write(qkv, hq, hk, dh, pos, _prep(inv, **dict(kw)), c1, slots)
        q2 = ref.qk_prepare_kv_write(qkv, hq, hk, dh, pos, _prep(inv, **dict(kw)), c2, slots)
        assert torch.allclose(q1.float(), q2.float(), **_tol(dt)), kw
        assert torch.allclose(c1.float(), c2.float(), **_tol(dt)), kw
    # the pairing matters: half-split and adjacent pairs give different rows
    a = ref.qk_prepare_kv_write(qkv, hq, hk, dh, pos, _prep(inv, pairing="half", rotary_dim=rd), None, None)
    b = ref.qk_prepare_kv_write(qkv, hq, hk, dh, pos, _prep(inv, pairing="adjacent", rotary_dim=rd), None, None)
    assert not torch.allclose(a.float(), b.float(), atol=1e-2)


def test_rotation_angles_are_float32_at_large_positions(ops):
    # the angle must be pos * inv_freq in float32: with a bfloat16 position 257 becomes 256
    dh = 16
    qkv = torch.zeros(1, 3 * dh, device=DEV)
    qkv[0, 0] = 1.0
    inv_freq = (1.0 / (10000.0 ** (torch.arange(0, dh, 2).float() / dh))).to(DEV)
    for p in (257, 4099, 131071):
        pos = torch.tensor([p], dtype=torch.int32, device=DEV)
        q = ops.qk_prepare_kv_write(qkv, 1, 1, dh, pos, _prep(inv_freq), None, None)
        assert abs(float(q[0, 0, 0]) - math.cos(float(torch.tensor(float(p)) * inv_freq[0].cpu()))) < 2e-6
        assert abs(float(q[0, 0, 1]) - math.sin(float(torch.tensor(float(p)) * inv_freq[0].cpu()))) < 2e-6


def _attention_case(hq, hk, dh, ps, dt, seg_specs, seed=0):
    """seg_specs: (tokens already in the cache, new tokens) per segment; pages are scattered."""
    g = torch.Generator().manual_seed(seed)
    total_pages = sum(-(-(a + b) // ps) for a, b in seg_specs) + 5
    perm = torch.randperm(total_pages, generator=g).tolist()
    kv = (torch.randn(total_pages, 2, hk, ps, dh, generator=g) * 0.7).to(dt).to(DEV)
    width = max(-(-(a + b) // ps) for a, b in seg_specs)
    bt = torch.full((len(seg_specs), width), -1, dtype=torch.int32)
    pos, seg = [], []
    for i, (a, b) in enumerate(seg_specs):
        for j in range(-(-(a + b) // ps)):
            bt[i, j] = perm.pop()
        pos += list(range(a, a + b))
        seg += [i] * b
    n = len(pos)
    q = (torch.randn(n, hq, dh, generator=g)).to(dt).to(DEV)
    return (q, kv, bt.to(DEV), torch.tensor(pos, dtype=torch.int32, device=DEV),
            torch.tensor(seg, dtype=torch.int32, device=DEV))


@pytest.mark.parametrize("dt", DT)
@pytest.mark.parametrize("hq,hk,dh,ps", [(4, 2, 16, 16), (5, 1, 48, 16), (6, 3, 32, 8), (8, 8, 64, 16),
                                         (10, 2, 128, 16), (2, 1, 256, 32), (3, 1, 80, 16), (6, 3, 32, 16),
                                         (40, 8, 128, 16), (20, 1, 96, 48), (4, 4, 256, 16), (5, 5, 64, 64),
                                         (10, 2, 128, 32), (9, 3, 128, 48), (10, 5, 128, 64)])
@pytest.mark.parametrize("retention", [("all",), ("chunk", 24), ("window", 37)])
def test_paged_attention(ops, ref, dt, hq, hk, dh, ps, retention):
    case = _attention_case(hq, hk, dh, ps, dt, [(0, 70), (130, 1), (45, 9), (63, 2), (200, 1), (600, 1), (255, 3)])
    q, kv, bt, pos, seg = case
    got = ops.paged_attention(q, kv, bt, pos, seg, retention, dh ** -0.5)
    want = ref.paged_attention(q, kv, bt, pos, seg, retention, dh ** -0.5)
    _assert_close_to_scale(got, want, dt)


@pytest.mark.parametrize("hq,hk,dh,ps", [(4, 2, 16, 16), (5, 1, 48, 16), (8, 8, 64, 16), (10, 2, 128, 16), (2, 1, 256, 32),
                                         (3, 1, 80, 16), (20, 1, 96, 48), (9, 3, 128, 48), (5, 5, 64, 64)])
@pytest.mark.parametrize("retention", [("all",), ("chunk", 24), ("chunk", 100), ("window", 37)])
def test_float32_attention_of_portions_on_the_float32_matrix_instructions(ops, ref, monkeypatch, hq, hk, dh, ps, retention):
    """Tiles of 16 tokens per wavefront (steps of many tokens in float32 take this kernel): portions that start
    anywhere, single tokens between them, keys of earlier steps; and a token's result does not depend on which
    tile it falls into."""
    monkeypatch.setattr(type(ops), "GENERIC_SPLIT_BELOW", 0)
    specs = [(0, 70), (130, 1), (45, 9), (63, 2), (200, 1), (600, 1), (255, 35)]
    q, kv, bt, pos, seg = _attention_case(hq, hk, dh, ps, torch.float32, specs)
    calls = []
    inner = ops._call
    monkeypatch.setattr(ops, "_call", lambda name, *a: (calls.append(name), inner(name, *a))[1])
    got = ops.paged_attention(q, kv, bt, pos, seg, retention, dh ** -0.5)
    assert calls == ["jle_attention_f32_tiles"]
    want = ref.paged_attention(q, kv, bt, pos, seg, retention, dh ** -0.5)
    _assert_close_to_scale(got, want, torch.float32)
    # the last 20 tokens of the last portion alone (other tiles, an odd start): the same bits
    n = q.shape[0]
    alone = ops.paged_attention(q[n - 20:].contiguous(), kv, bt, pos[n - 20:].contiguous(), seg[n - 20:].contiguous(),
                                retention, dh ** -0.5)
    assert torch.equal(alone, got[n - 20:])


@pytest.mark.parametrize("hq,hk,dh,ps", [(4, 2, 16, 16), (5, 1, 48, 16), (40, 8, 128, 16), (16, 1, 64, 32), (3, 3, 256, 16)])
@pytest.mark.parametrize("retention", [("all",), ("chunk", 100), ("window", 37)])
def test_float32_attention_of_single_tokens_on_the_float32_matrix_instructions(ops, ref, monkeypatch, hq, hk, dh, ps, retention):
    """A step of single tokens in float32: the query heads of a kv head share a wavefront, the keys are shared
    between wavefronts (forced here to ranges of 64 keys, so that every token has several) and merged."""
    monkeypatch.setattr(type(ops), "F32_DECODE_ITEMS", 1 << 20)
    specs = [(130, 1), (0, 1), (63, 1), (200, 1), (600, 1), (15, 1), (99, 1)]
    q, kv, bt, pos, seg = _attention_case(hq, hk, dh, ps, torch.float32, specs)
    calls = []
    inner = ops._call
    monkeypatch.setattr(ops, "_call", lambda name, *a: (calls.append(name), inner(name, *a))[1])
    got = ops.paged_attention(q, kv, bt, pos, seg, retention, dh ** -0.5)
    assert calls == ["jle_attention_f32_heads", "jle_attention_merge"]
    want = ref.paged_attention(q, kv, bt, pos, seg, retention, dh ** -0.5)
    _assert_close_to_scale(got, want, torch.float32)
    monkeypatch.setattr(type(ops), "F32_DECODE_ITEMS", 1)  # one range per token: no merge
    calls.clear()
    whole = ops.paged_attention(q, kv, bt, pos, seg, retention, dh ** -0.5)
    assert calls == ["jle_attention_f32_heads"]
    _assert_close_to_scale(whole, want, torch.float32)


@pytest.mark.parametrize("hq,hk,ps", [(10, 2, 16), (40, 8, 16), (6, 3, 32), (9, 3, 48), (4, 2, 64)])
@pytest.mark.parametrize("retention", [("all",), ("chunk", 192), ("chunk", 100), ("window", 150)])
def test_paged_attention_of_long_portions_at_head_size_128(ops, ref, hq, hk, ps, retention):
    """Portions of hundreds of tokens behind hundreds of cached ones, at the head size whose kernel takes 64 keys a
    step straight into shared memory: many steps, pages of every size crossed inside a step, rules whose first
    key lies inside a step and inside a page."""
    dt = torch.bfloat16
    case = _attention_case(hq, hk, 128, ps, dt, [(0, 333), (190, 130), (517, 1), (64, 64), (1000, 35)], seed=3)
    q, kv, bt, pos, seg = case
    got = ops.paged_attention(q, kv, bt, pos, seg, retention, 128 ** -0.5)
    want = ref.paged_attention(q, kv, bt, pos, seg, retention, 128 ** -0.5)
    _assert_close_to_scale(got, want, dt)


@pytest.mark.parametrize("hq,hk,dh,ps", [(10, 2, 128, 16), (16, 8, 128, 48), (3, 3, 64, 16), (4, 2, 64, 64), (6, 3, 64, 8)])
@pytest.mark.parametrize("window,keep", [(150, 5), (70, 64), (64, 65), (1, 1), (33, 0), (2000, 8)])
@pytest.mark.parametrize("shared", [0, 1 << 20])
def test_single_tokens_with_kept_ones_at_the_edges_of_tiles(ops, ref, monkeypatch, hq, hk, dh, ps, window, keep, shared):
    """Whole tiles' loads asked for ahead (64 and 128 elements, pages of sixteens; another page size for the other form): last
    keys at the edges of sixteens, tiles and pages, windows and kept ranges that begin and end inside them, a query's keys in
    one wavefront and shared.  Slots that no query sees are poisoned, pages of nothing else are given back, and a token whose
    own page is missing gets NaN."""
    monkeypatch.setattr(type(ops), "GENERIC_SPLIT_BELOW", shared)
    dt = torch.bfloat16
    ends = [0, 1, 15, 16, 31, 47, 48, 63, 64, 65, 127, 128, 191, 250, 600]
    q, kv, bt, pos, seg = _attention_case(hq, hk, dh, ps, dt, [(a, 1) for a in ends], seed=5)
    want = ref.paged_attention(q, kv, bt, pos, seg, ("window_keep", window, keep), dh ** -0.5)
    for i, a in enumerate(ends):
        first = max(0, a - window + 1)
        for j in range(-(-(a + 1) // ps)):
            page = int(bt[i, j])
            for o in range(ps):
                if j * ps + o > a or keep <= j * ps + o < first:
                    kv[page, 0].view(hk, ps, dh)[:, o] = float("nan")
                    kv[page, 1].view(hk, dh, ps)[:, :, o] = float("nan")  # (values lie transposed)
            if keep <= j * ps and (j + 1) * ps <= first:
                bt[i, j] = -1
    calls = []
    inner = ops._call
    monkeypatch.setattr(ops, "_call", lambda name, *a: (calls.append(name), inner(name, *a))[1])
    got = ops.paged_attention(q, kv, bt, pos, seg, ("window_keep", window, keep), dh ** -0.5)
    assert calls == ["jle_paged_attention_kept"]
    _assert_close_to_scale(got, want, dt)
    bt[-1, 600 // ps] = -1
    gone = ops.paged_attention(q, kv, bt, pos, seg, ("window_keep", window, keep), dh ** -0.5)
    assert torch.isnan(gone[-1]).all() and torch.equal(gone[:-1], got[:-1])


@pytest.mark.parametrize("hq,hk,ps", [(10, 2, 16), (16, 8, 16), (9, 3, 48), (4, 2, 64), (3, 3, 16)])
@pytest.mark.parametrize("window,keep", [(150, 5), (70, 64), (64, 65), (100, 200), (1, 1), (33, 0), (2000, 8)])
def test_attention_with_kept_tokens_of_long_portions_at_head_size_128(ops, ref, monkeypatch, hq, hk, ps, window, keep):
    """Kept keys in steps of their own before the window's, beside it and within it, kept ranges that end inside a step and
    inside a page, portions that lie before, across and behind the window's first move, a single token between them.  Pages
    that no query sees are given back, and what lies beside the visible keys of the others is poisoned."""
    dt = torch.bfloat16
    specs = [(0, 333), (190, 130), (517, 1), (64, 64), (1000, 35)]
    q, kv, bt, pos, seg = _attention_case(hq, hk, 128, ps, dt, specs, seed=3)
    want = ref.paged_attention(q, kv, bt, pos, seg, ("window_keep", window, keep), 128 ** -0.5)
    for i, (a, b) in enumerate(specs):
        first = max(0, a - window + 1)
        for j in range(-(-(a + b) // ps)):
            page = int(bt[i, j])
            for o in range(ps):
                if j * ps + o >= a + b or keep <= j * ps + o < first:
                    kv[page, 0, :, o] = float("nan")
                    kv[page, 1].view(hk, 128, ps)[:, :, o] = float("nan")  # (values lie transposed)
            if keep <= j * ps and (j + 1) * ps <= first:
                bt[i, j] = -1
    calls = []
    inner = ops._call
    monkeypatch.setattr(ops, "_call", lambda name, *a: (calls.append(name), inner(name, *a))[1])
    got = ops.paged_attention(q, kv, bt, pos, seg, ("window_keep", window, keep), 128 ** -0.5)
    assert calls == ["jle_attention_prefill_kept"]
    _assert_close_to_scale(got, want, dt)


@pytest.mark.parametrize("window,keep,n", [(1024, 8, 80), (150, 70, 1111), (1024, 8, 2048)])
def test_keys_shared_between_wavefronts_lose_no_precision(ops, window, keep, n):
    """Query heads that share kv heads against the same kv heads given to each (whose wavefronts read their own keys): both
    take a running maximum every 32 keys and round the same probabilities, so that only the orders of float32 sums differ."""
    q, kv, bt, pos, seg = _attention_case(8, 4, 128, 16, torch.bfloat16, [(0, n)], seed=11)
    pages, twice = bt[0].long(), kv.repeat_interleave(2, dim=2)
    keys = twice[pages, 0].permute(1, 0, 2, 3).reshape(8, -1, 128)[:, :n].double()
    values = twice[pages, 1].reshape(-1, 8, 128, 16).permute(1, 0, 3, 2).reshape(8, -1, 128)[:, :n].double()  # (stored transposed)
    at = torch.arange(n, device=DEV)
    hidden = (at[None] > at[:, None]) | (at[:, None] - at[None] >= window) & (at[None] >= keep)
    want = torch.stack([torch.softmax((q[:, h].double() @ keys[h].T.contiguous() * 128 ** -0.5).masked_fill(hidden, -math.inf), -1) @ values[h]
                        for h in range(8)], 1)
    err = [float((ops.paged_attention(q, pool, bt, pos, seg, ("window_keep", window, keep), 128 ** -0.5).view(n, 8, 128).double() - want).norm())
           for pool in (kv, twice)]
    assert err[0] <= 1.001 * err[1]


def test_attention_with_kept_tokens_of_layers_with_other_heads_in_one_step(ops, ref):
    """Layers of one step with other numbers of heads find lists laid out for their own; window and kept range change none."""
    import types

    ctx = types.SimpleNamespace(meta={}, seg_lens=[100, 70], seg_starts=[0, 300], decode_bucket=None)
    for hq, hk, retention in ((16, 8, ("window_keep", 90, 5)), (12, 2, ("window_keep", 90, 5)), (4, 2, ("window_keep", 90, 5)),
                              (16, 8, ("window_keep", 33, 70))):
        q, kv, bt, pos, seg = _attention_case(hq, hk, 128, 16, torch.bfloat16, [(0, 100), (300, 70)], seed=hq)
        got = ops.paged_attention(q, kv, bt, pos, seg, retention, 128 ** -0.5, meta=ctx)
        _assert_close_to_scale(got, ref.paged_attention(q, kv, bt, pos, seg, retention, 128 ** -0.5), torch.bfloat16)


@pytest.mark.parametrize("n,d,e,k,experts,groups", [
    (5, 1032, 2, 1, 2, None), (5, 2048, 10, 2, 8, (5, 3)), (8, 2056, 16, 8, 16, (4, 2)), (16, 2048, 9, 4, 8, None),
    (17, 4096, 16, 3, 12, (8, 5)), (32, 2048, 10, 2, 8, (5, 3)), (64, 8192, 8, 1, 8, None), (64, 4096, 16, 1, 16, (2, 1)),
    (8, 4104, 9, 2, 8, None), (9, 4104, 9, 2, 8, None), (16, 8192, 16, 4, 12, (4, 2))])
@pytest.mark.parametrize("extra", [False, True])
def test_choices_by_scores_token_by_token_equal_the_separate_kernels(ops, monkeypatch, n, d, e, k, experts, groups, extra):
    """A block a token with all its experts (up to 16, up to 64 choices): the bits of norm, logits, choice and grouping as
    launches of their own, launch after launch, with equal scores, a token that is not finite and identity experts."""
    x, w, router = _rand(n, d, seed=1), _rand(d, seed=2) + 1.0, _rand(e, d, scale=0.05, seed=3)
    router[e - 1] = router[0]
    delta = _rand(n, d, dt=torch.bfloat16, seed=4)
    x[n - 1, 3] = float("inf")
    correction = _rand(e, scale=0.1, seed=5)
    g, keep = groups or (None, None)
    calls = []
    inner = ops._call
    for scores in ("sigmoid", "softmax"):
        args = dict(groups=g, keep_groups=keep, group_terms=1, scores=scores, normalize=1e-20 if extra else None, weight_scale=1.5,
                    num_experts=experts, extra_group=extra)
        for _ in range(2):
            with monkeypatch.context() as m:
                m.setattr(ops, "_call", lambda name, *a: (calls.append(name), inner(name, *a))[1])
                pending = ops.defer_norm(x.clone(), delta, w, 1e-5, torch.bfloat16)
                ids, weights, grouping = ops.moe_choose(pending, router, correction, k, **args)
            assert calls[-1] == "jle_norm_route"
            h, h32 = ops.add_rmsnorm(x.clone(), delta, w, 1e-5, torch.bfloat16, want32=True)
            want = ops.moe_choose(h32, router, correction, k, **args)
            ok = torch.arange(n, device=DEV) < n - 1  # (the last token's numbers are NaN: any order will do, its rows exist)
            assert torch.equal(ids[ok], want[0][ok]) and torch.equal(weights[ok], want[1][ok])
            assert torch.equal(pending.rows()[ok], h[ok]) and bool(((ids >= 0) & (ids < e)).all())
            off, tok, gate, inv = (t.cpu() for t in grouping)
            again = [t.cpu() for t in ops.moe_align(ids, weights, experts, extra_group=len(off) == experts + 2, note_extra=True)]
            rows = int(again[0][-1])  # (behind them nothing is written: identity experts)
            assert torch.equal(off, again[0]) and torch.equal(inv, again[3]) and torch.equal(tok[:rows], again[1][:rows])
            assert torch.equal(gate[:rows].view(torch.int32), again[2][:rows].view(torch.int32))


@pytest.mark.parametrize("n,d,e,k,experts,groups", [
    (1, 4, 1, 1, 1, None), (1, 2048, 10, 2, 8, (5, 3)), (16, 2052, 4, 4, 3, None), (17, 1020, 5, 1, 5, None), (32, 2048, 8, 2, 8, (4, 2)),
    (33, 2048, 8, 2, 8, (4, 2)), (64, 4100, 9, 2, 7, None), (65, 2048, 16, 2, 16, (4, 2)), (128, 512, 16, 2, 12, (8, 5)),
    (129, 2048, 8, 2, 8, None), (200, 256, 16, 16, 16, None), (256, 2048, 10, 1, 8, None), (257, 2048, 10, 1, 8, None),
    (15, 4096, 10, 2, 8, None), (64, 4096, 16, 4, 16, None)])
@pytest.mark.parametrize("extra", [False, True])
def test_router_and_choice_in_one_launch_equal_the_separate_kernels(ops, monkeypatch, n, d, e, k, experts, groups, extra):
    """A block a token with all its experts: the bits of logits and choice as launches of their own, at the edges of a
    wavefront's experts, of the pieces of a row and of the pairs that one wavefront groups; the grouping against a stable sort."""
    h, router, correction = _rand(n, d, seed=1), _rand(e, d, scale=0.05, seed=2), _rand(e, scale=0.1, seed=3)
    router[e - 1] = router[0]
    g, keep = groups or (None, None)
    calls = []
    inner = ops._call
    monkeypatch.setattr(ops, "_call", lambda name, *a: (calls.append(name), inner(name, *a))[1])
    for scores, corr in (("sigmoid", correction), ("softmax", None)):
        args = dict(groups=g, keep_groups=keep, group_terms=1, scores=scores, normalize=1e-20 if extra else None, weight_scale=1.5,
                    num_experts=experts, extra_group=extra)
        calls.clear()
        ids, weights, grouping = ops.moe_choose(h, router, corr, k, **args)
        assert calls[0] == ("jle_moe_logits" if (n, d, e) in ((257, 2048, 10), (15, 4096, 10), (64, 4096, 16)) else "jle_moe_logits_choose")
        with monkeypatch.context() as m:
            m.setattr(type(ops), "CHOOSE_TOKENS", 0)
            want = ops.moe_choose(h, router, corr, k, **args)
        assert torch.equal(ids, want[0]) and torch.equal(weights, want[1])
        assert all(a.shape == b.shape for a, b in zip(grouping, want[2]))
        off, tok, gate, inv = (t.cpu() for t in grouping)
        flat = ids.cpu().reshape(-1)
        order = [int(r) for r in torch.argsort(flat, stable=True) if flat[r] < experts]
        counts = torch.bincount(flat.long(), minlength=e)[:experts]
        assert off[: experts + 1].tolist() == [0, *torch.cumsum(counts, 0).tolist()]
        assert tok[: len(order)].tolist() == [r // k for r in order]
        assert torch.equal(gate[: len(order)], weights.cpu().reshape(-1)[order])
        ld = inv.numel() // n
        row = {r: i for i, r in enumerate(order)}
        assert inv.view(n, ld)[:, :k].reshape(-1).tolist() == [row.get(r, -1) for r in range(n * k)]
        if len(off) == experts + 2:  # (a shared expert's rows behind the others)
            assert int(off[-1]) == len(order) + n and tok[len(order): len(order) + n].tolist() == list(range(n))
            assert ld == k + 1 and inv.view(n, ld)[:, k].tolist() == [len(order) + t for t in range(n)]
            assert bool((gate[len(order): len(order) + n] == 1).all())


class _Segments:
    """What the matrix-memory kernels read of a step."""

    def __init__(self, seg_lens, slots, phases):
        cu = [0]
        for ln in seg_lens:
            cu.append(cu[-1] + ln)
        ints = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)
        self.seg_lens, self.num_segments, self.num_tokens = list(seg_lens), len(seg_lens), cu[-1]
        self.cu_seqlens, self.state_slots, self.state_phase = ints(cu), ints(slots), ints(phases)
        self.scratch = {}


def _matrix_memory_float64(rows, gates, b_gates, norm_w, H, dk, dv, cap, eps, floor, state, seg_lens, slots, phases):
    """The recurrence written out, float64 on the host: outputs [N, H dv] and the states behind every segment."""
    rows, gates, b_gates, norm_w, state = (t.double().cpu() for t in (rows, gates, b_gates, norm_w, state))
    n = rows.shape[0]
    q = rows[:, : H * dk].reshape(n, H, dk) * dk ** -0.5
    k = rows[:, H * dk: 2 * H * dk].reshape(n, H, dk)
    v = rows[:, 2 * H * dk: 2 * H * dk + H * dv].reshape(n, H, dv)
    z = cap * torch.tanh((gates + b_gates) / cap)
    li, lf = z[:, :H], torch.nn.functional.logsigmoid(z[:, H:])
    out = torch.zeros(n, H, dv, dtype=torch.float64)
    new_state = state.clone()
    t = 0
    for ln, slot, ph in zip(seg_lens, slots, phases):
        st = state[slot, ph]
        C, nn_, m = st[:, : dk * dv].reshape(H, dk, dv).clone(), st[:, dk * dv: dk * dv + dk].clone(), st[:, -1].clone()
        for _ in range(ln):
            m2 = torch.maximum(lf[t] + m, li[t])
            keep, take = torch.exp(lf[t] + m - m2), torch.exp(li[t] - m2)
            C = keep[:, None, None] * C + take[:, None, None] * k[t][:, :, None] * v[t][:, None, :]
            nn_ = keep[:, None] * nn_ + take[:, None] * k[t]
            m = m2
            den = torch.maximum((nn_ * q[t]).sum(-1).abs(), torch.exp(-m)) + floor
            out[t] = torch.einsum("hkv,hk->hv", C, q[t]) / den[:, None]
            t += 1
        new_state[slot, 1 - ph] = torch.cat([C.reshape(H, dk * dv), nn_, m[:, None]], dim=1)
    o = out / torch.sqrt(out.pow(2).mean(-1, keepdim=True) + eps)
    o = o.reshape(n, H * dv) * norm_w * torch.sigmoid(rows[:, 2 * H * dk + H * dv:])
    return o, new_state


@pytest.mark.parametrize("dt", DT)
@pytest.mark.parametrize("H,dk,dv", [(2, 16, 16), (3, 24, 40), (1, 10, 6), (4, 64, 128), (2, 128, 64), (2, 7, 70), (1, 100, 130)])
@pytest.mark.parametrize("gates_at", ["middle", "forgetting", "keeping"])
def test_matrix_memory_in_chunks_equals_token_by_token(ops, ref, monkeypatch, dt, H, dk, dv, gates_at):
    """Segments that end before, at and behind a chunk's edge, single tokens beside them, states that are not zero
    and whose running maximum is far from the gates, slots in any order and either half: the chunked kernels
    against the plain recurrence, outputs and new states; and the same step without chunks."""
    seg_lens = [200, 1, 64, 7, 65, 1, 63, 128, 9]
    ctx = _Segments(seg_lens, slots=[3, 0, 8, 5, 1, 7, 2, 4, 6], phases=[0, 1, 1, 0, 0, 1, 0, 1, 0])
    n = ctx.num_tokens
    g = torch.Generator().manual_seed(H * 100 + dk)
    rows = (torch.randn(n, 2 * H * dk + 2 * H * dv, generator=g)).to(dt).to(DEV)
    shift = {"middle": 0.0, "forgetting": -6.0, "keeping": 9.0}[gates_at]
    gates = (torch.randn(n, 2 * H, generator=g) * 3.0).to(DEV)
    gates[:, H:] += shift
    b_gates = torch.randn(2 * H, generator=g).to(DEV)
    norm_w = (torch.rand(H * dv, generator=g) + 0.5).to(DEV)
    state = torch.randn(9, 2, H, dk * dv + dk + 1, generator=g).to(DEV)
    state[:, :, :, -1] = torch.randn(9, 2, H, generator=g).to(DEV) * 8.0  # running maxima
    st_got, st_scan = state.clone(), state.clone()
    slots, phases = ctx.state_slots.tolist(), ctx.state_phase.tolist()
    want, st_ref = _matrix_memory_float64(rows, gates, b_gates, norm_w, H, dk, dv, 9.0, 1e-5, 1e-6, state, seg_lens,
                                          slots, phases)
    calls = []
    inner = ops._call
    monkeypatch.setattr(ops, "_call", lambda name, *a: (calls.append(name), inner(name, *a))[1])
    got = ops.mlstm(rows, gates.clone(), b_gates, norm_w, H, dk, dv, 9.0, 1e-5, 1e-6, st_got, ctx)
    assert calls == ["jle_mlstm_chunked"]
    monkeypatch.setattr(type(ops), "MLSTM_CHUNKS_FROM", 10 ** 9)
    scan = ops.mlstm(rows, gates.clone(), b_gates, norm_w, H, dk, dv, 9.0, 1e-5, 1e-6, st_scan, ctx)
    assert calls[-1] == "jle_mlstm"
    # (under strong forgetting n . q can be a small difference of large terms: the token-by-token kernel's float32
    # sums then lose a digit more than the chunks' sums on the matrix instruction)
    for name, other, tol32 in (("chunks", got, 1e-4), ("token by token", scan, 1e-3)):
        assert torch.isfinite(other).all(), name
        err = float((other.double().cpu() - want).abs().max())
        assert err < (tol32 if dt == torch.float32 else 2e-2), (name, err)
    for name, st in (("chunks", st_got), ("token by token", st_scan)):
        for slot, ph in zip(slots, phases):  # the halves that the step wrote
            a, b = st[slot, 1 - ph].double().cpu(), st_ref[slot, 1 - ph]
            assert float(((a - b).abs() / b.abs().amax(dim=-1, keepdim=True).clamp_min(1.0)).max()) < 1e-5, (name, slot)
            assert torch.equal(st[slot, ph], state[slot, ph]), "the half that the step reads stays as it was"


def _distance_table(hq, length, seed):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(hq, length, generator=g) * 1.5).to(DEV)


@pytest.mark.parametrize("dt", DT)
@pytest.mark.parametrize("hq,hk,dh,ps", [(4, 2, 16, 16), (8, 2, 64, 16), (10, 2, 128, 16), (5, 1, 96, 48), (3, 3, 32, 32),
                                         (34, 2, 32, 16), (2, 1, 256, 16), (6, 3, 80, 16)])
@pytest.mark.parametrize("length,with_sink", [(1, True), (9, True), (41, False), (130, True), (700, True)])
def test_attention_with_distance_bias_and_sinks(ops, ref, monkeypatch, dt, hq, hk, dh, ps, length, with_sink):
    """Portions and single tokens in one step, with a table that ends before, inside and beyond the contexts, keys
    ranges of a single token that are merged, and a sink per head that is larger or smaller than the scores."""
    specs = [(0, 70), (130, 1), (45, 9), (63, 2), (200, 1), (600, 1), (255, 35), (0, 1)]
    q, kv, bt, pos, seg = _attention_case(hq, hk, dh, ps, dt, specs, seed=2)
    bias = _distance_table(hq, length, seed=length)
    sink = (torch.linspace(-6.0, 7.0, hq)).to(DEV) if with_sink else None
    calls = []
    inner = ops._call
    monkeypatch.setattr(ops, "_call", lambda name, *a: (calls.append(name), inner(name, *a))[1])
    got = ops.paged_attention(q, kv, bt, pos, seg, ("all",), dh ** -0.5, bias=bias, sink=sink)
    if dt == torch.bfloat16 and dh in (32, 64, 96, 128, 256):
        assert calls == ["jle_attention_prefill", "jle_attention_decode"]
    want = ref.paged_attention(q, kv, bt, pos, seg, ("all",), dh ** -0.5, bias=bias, sink=sink)
    _assert_close_to_scale(got, want, dt)
    if with_sink:  # a sink alone
        got = ops.paged_attention(q, kv, bt, pos, seg, ("all",), dh ** -0.5, sink=sink)
        want = ref.paged_attention(q, kv, bt, pos, seg, ("all",), dh ** -0.5, sink=sink)
        _assert_close_to_scale(got, want, dt)


@pytest.mark.parametrize("hq,hk,ps", [(10, 2, 16), (16, 8, 16), (6, 3, 32), (9, 3, 48), (4, 2, 64)])
@pytest.mark.parametrize("length", [1, 70, 400, 1300])
def test_biased_attention_of_long_portions_at_head_size_128(ops, ref, hq, hk, ps, length):
    """The kernel that shares a step's keys between the wavefronts of a block, with a distance table and sinks:
    portions of hundreds of tokens behind hundreds of cached ones, tables that end inside a step of 64 keys, before
    the portion and beyond every context."""
    dt = torch.bfloat16
    q, kv, bt, pos, seg = _attention_case(hq, hk, 128, ps, dt, [(0, 333), (190, 130), (517, 1), (64, 64), (1000, 35)], seed=3)
    bias = _distance_table(hq, length, seed=length + 1)
    sink = torch.linspace(-4.0, 6.0, hq).to(DEV)
    got = ops.paged_attention(q, kv, bt, pos, seg, ("all",), 128 ** -0.5, bias=bias, sink=sink)
    want = ref.paged_attention(q, kv, bt, pos, seg, ("all",), 128 ** -0.5, bias=bias, sink=sink)
    _assert_close_to_scale(got, want, dt)


@pytest.mark.parametrize("dh", [64, 128])
@pytest.mark.parametrize("back", [0, 1, 30, 31, 32, 63, 64, 65, 200])
def test_a_distance_table_entry_that_stands_out_picks_its_key(ops, ref, dh, back):
    """One entry of the table is so large that the key that many places back takes the whole weight, in a portion
    and in a single token with merged key ranges; in the table's last entry every key from there on shares it.
    With all queries zero the scores are the table's alone."""
    dt = torch.bfloat16
    hq, hk, ps, length = 4, 2, 16, 65
    q, kv, bt, pos, seg = _attention_case(hq, hk, dh, ps, dt, [(100, 250), (2000, 1), (3, 40)], seed=4)
    q = torch.zeros_like(q)
    bias = torch.zeros(hq, length, device=DEV)
    bias[:, min(back, length - 1)] = 60.0
    got = ops.paged_attention(q, kv, bt, pos, seg, ("all",), dh ** -0.5, bias=bias).float().view(-1, hq, dh)
    vt = kv[:, 1].reshape(kv.shape[0], hk, dh, ps).float()  # (the value planes lie transposed)
    for i in (0, 17, 249, 250, 251, 290):
        p, sg = int(pos[i]), int(seg[i])
        firsts = [p - back] if back < length - 1 else list(range(0, p - length + 2))
        firsts = [k for k in firsts if k >= 0]
        if not firsts:
            continue
        rows = torch.stack([vt[int(bt[sg, k // ps]), :, :, k % ps] for k in firsts]).mean(dim=0)  # [hk, dh]
        want = rows.repeat_interleave(hq // hk, dim=0)
        assert torch.allclose(got[i], want, atol=2e-2), (i, back)


def _decode_case(hq, hk, dh, ps, dt, contexts, seed=0):
    """One new token per request after ``contexts[i]`` tokens in the cache; the step's group context with the
    bound the kernels' work is laid out for; raw q|k|v rows and the slots of the new tokens."""
    from jax_llm_examples_amd.engine.batch import GroupContext, decode_bucket
    q, kv, bt, pos, seg = _attention_case(hq, hk, dh, ps, dt, [(c, 1) for c in contexts], seed=seed)
    n = len(contexts)
    g = torch.Generator().manual_seed(seed + 50)
    qkv = torch.randn(n, (hq + 2 * hk) * dh, generator=g).to(dt).to(DEV)
    slots = torch.tensor([int(bt[i, c // ps]) * ps + c % ps for i, c in enumerate(contexts)], dtype=torch.int32,
                         device=DEV)
    meta = lambda ret: GroupContext(block_table=bt, slot_mapping=slots, width=bt.shape[1], retention=ret,
                                    seg_lens=[1] * n, seg_starts=list(contexts),
                                    decode_bucket=decode_bucket(max(contexts) + 1))
    return qkv, kv, bt, pos, seg, slots, meta


_DECODE_CASES = [
    (40, 8, 128, 16, [3000 + 94 * i for i in range(64)]),  # the serving shape: 64 requests between 3,000 and 9,000
    (40, 8, 128, 16, [8191, 8192, 8193, 0, 5, 16383, 16384, 4095]),
    (10, 2, 64, 32, [0, 1, 31, 32, 700, 129]), (6, 1, 32, 16, [77]), (20, 1, 96, 48, [500, 47, 48]),
    (34, 2, 32, 16, [260, 3]), (4, 4, 256, 16, [90, 1000])]
_DECODE_RETENTIONS = [("all",), ("chunk", 8192), ("chunk", 96), ("window", 200)]


@pytest.mark.parametrize("dt", DT)
@pytest.mark.parametrize("hq,hk,dh,ps,contexts,retention",
                         [(*c, r) for c in _DECODE_CASES for r in _DECODE_RETENTIONS
                          if r != ("chunk", 8192) or max(c[4]) >= 3000])  # (the large chunk: long contexts only)
def test_attention_of_a_step_of_single_tokens_from_the_projection_rows(ops, ref, dt, hq, hk, dh, ps, contexts, retention):
    """Rotation, q/k norm, scale, the write of the new key and value, attention over many key ranges and their
    merge: one launch in bfloat16 (two kernels and a merge in float32), against the plain ops."""
    from jax_llm_examples_amd.ops.hip import HipOps
    qkv, kv, bt, pos, seg, slots, meta = _decode_case(hq, hk, dh, ps, dt, contexts)
    inv = (1.0 / (10000.0 ** (torch.arange(0, dh, 2).float() / dh))).to(DEV)
    for prep in (_prep(inv, 1e-5, None), _prep(None, None, (64.0, 0.2)), _prep(inv, None, None)):
        kv1, kv2 = kv.clone(), kv.clone()
        calls = []
        inner = ops._call
        ops._call = lambda name, *a: (calls.append(name), inner(name, *a))[1]
        try:
            got = ops.attention_from_qkv(qkv, hq, hk, dh, pos, seg, prep, kv1, True, slots, bt, retention,
                                         dh ** -0.5, meta(retention))
        finally:
            ops._call = inner
        if dt == torch.bfloat16:
            assert calls == ["jle_attention_decode_fused"], calls
        want = ref.attention_from_qkv(qkv, hq, hk, dh, pos, seg, prep, kv2, True, slots, bt, retention, dh ** -0.5)
        _assert_close_to_scale(got, want, dt)
        assert torch.allclose(kv1.float(), kv2.float(), **_tol(dt))  # the new keys and values are in their pages
        assert int(ops._tickets.abs().sum()) == 0  # the counters are back at zero
        # a run that only reads another run's cache writes nothing
        kv3 = kv2.clone()
        got3 = ops.attention_from_qkv(qkv, hq, hk, dh, pos, seg, prep, kv3, False, slots, bt, retention,
                                      dh ** -0.5, meta(retention))
        assert torch.equal(kv3, kv2)
        _assert_close_to_scale(got3, want, dt)


@pytest.mark.parametrize("dt", DT)
def test_decode_attention_finds_a_far_key_in_every_key_range_and_at_the_chunk_edge(ops, dt):
    """Eight requests around 8,200 tokens: so many key ranges that the work list is longer than the GPU takes at
    once.  One key's score stands out; the output is its value exactly where the rule lets the query see it."""
    hq, hk, dh, ps = 40, 8, 128, 16
    contexts = [8190 + i for i in range(8)]  # positions 8190 .. 8197
    qkv, kv, bt, pos, seg, slots, meta = _decode_case(hq, hk, dh, ps, dt, contexts, seed=2)
    qkv.zero_()
    qkv[:, : hq * dh].view(len(contexts), hq, dh)[:, :, 0] = 8.0  # every query looks along element 0
    prep = _prep(None, None, None)
    kv[:, 0] *= 0.05
    kv[:, 0, :, :, 0] = 0.0

    def run(hot, retention):
        k = kv.clone()
        for i in range(len(contexts)):
            page, off = int(bt[i, hot // ps]), hot % ps
            k[page, 0, :, off, 0] = 8.0
            k[page, 1].view(hk, dh, ps)[:, :, off] = 3.0
        out = ops.attention_from_qkv(qkv, hq, hk, dh, pos, seg, prep, k, False, slots, bt, retention, 1.0,
                                     meta(retention))
        return [bool(v > 2.9) for v in out.float().abs().amin(dim=-1).tolist()]

    for hot in (0, 127, 128, 511, 512, 4100, 8063, 8189):  # first and last range, range edges
        assert run(hot, ("all",)) == [True] * 8, hot
    assert run(8191, ("all",)) == [c >= 8191 for c in contexts]  # causal
    assert run(8191, ("chunk", 8192)) == [c == 8191 for c in contexts]  # the last key of the first chunk
    assert run(8192, ("chunk", 8192)) == [c >= 8192 for c in contexts]  # the first key of the second
    assert run(8000, ("chunk", 8192)) == [c < 8192 for c in contexts]
    assert run(8190 - 299, ("window", 300)) == [c == 8190 for c in contexts]


def test_attention_refuses_a_head_size_it_cannot_do(ops):
    from jax_llm_examples_amd.ops.hip import KernelError
    q, kv, bt, pos, seg = _attention_case(2, 1, 20, 16, torch.float32, [(0, 4)])
    with pytest.raises(KernelError, match="head size 20 is not supported"):
        ops.paged_attention(q, kv, bt, pos, seg, ("all",), 1.0)
    with pytest.raises(KernelError, match="top_k 9"):
        ops.moe_route(torch.zeros(2, 64, device=DEV), torch.zeros(16, 64, device=DEV), 9)


@pytest.mark.parametrize("dt", DT)
def test_attention_finds_one_far_key_among_hundreds_and_respects_the_window_edge(ops, dt):
    """Random weights would hide a key that is skipped: here one key's score stands out, so the
    output is that key's value, if and only if the rule lets the query see it."""
    hq, hk, dh, ps = 2, 1, 32, 16
    T = 700
    q, kv, bt, pos, seg = _attention_case(hq, hk, dh, ps, dt, [(T - 1, 1)], seed=3)
    q.zero_()
    q[0, :, 0] = 8.0

    def run(hot, retention):
        k = kv.clone()
        k[:, 0] *= 0.05
        page, off = int(bt[0, hot // ps]), hot % ps
        k[page, 0, 0, off, 0] = 8.0  # score 64 * scale, far above the rest
        k[page, 1, 0].view(dh, ps)[:, off] = 3.0  # its value (values lie transposed in the page)
        return ops.paged_attention(q, k, bt, pos, seg, retention, 1.0).float()

    for hot in (3, 15, 16, 17, 333, T - 2):  # page edges among them
        assert torch.allclose(run(hot, ("all",)), torch.full((1, hq * dh), 3.0, device=DEV), atol=2e-2)
    C = 96  # the query at 699 is in the chunk that starts at 672
    assert torch.allclose(run(672, ("chunk", C)), torch.full((1, hq * dh), 3.0, device=DEV), atol=2e-2)
    assert run(671, ("chunk", C)).abs().max() < 1.0  # one before the chunk: not seen
    W = 100  # window: keys 600..699
    assert torch.allclose(run(600, ("window", W)), torch.full((1, hq * dh), 3.0, device=DEV), atol=2e-2)
    assert run(599, ("window", W)).abs().max() < 1.0


@pytest.mark.parametrize("dt", DT)
def test_attention_portion_sees_a_far_key_exactly_where_the_rule_allows(ops, dt):
    """The same with a portion of 40 tokens (positions 660..699) in one step: with a chunk of 96 the tokens
    before 672 are in the chunk that starts at 576, the others in the one that starts at 672; with a window
    of 100 each token has its own edge."""
    hq, hk, dh, ps = 4, 2, 32, 16
    q, kv, bt, pos, seg = _attention_case(hq, hk, dh, ps, dt, [(660, 40)], seed=4)
    q.zero_()
    q[:, :, 0] = 8.0

    def run(hot, retention):
        k = kv.clone()
        k[:, 0] *= 0.05
        page, off = int(bt[0, hot // ps]), hot % ps
        k[page, 0, :, off, 0] = 8.0
        k[page, 1].view(hk, dh, ps)[:, :, off] = 3.0
        return ops.paged_attention(q, k, bt, pos, seg, retention, 1.0).float().abs().amin(dim=-1)  # per token

    def sees(out):
        return [bool(v > 2.9) for v in out.tolist()]

    assert sees(run(5, ("all",))) == [True] * 40
    assert sees(run(576, ("chunk", 96))) == [p < 672 for p in range(660, 700)]
    assert sees(run(575, ("chunk", 96))) == [False] * 40
    assert sees(run(672, ("chunk", 96))) == [p >= 672 for p in range(660, 700)]  # causal: not before its own position
    assert sees(run(580, ("window", 100))) == [p - 99 <= 580 for p in range(660, 700)]


def test_attention_reading_a_page_that_was_given_back_is_not_silent(ops):
    q, kv, bt, pos, seg = _attention_case(2, 1, 16, 16, torch.float32, [(40, 1)])
    bt[0, 1] = -1
    out = ops.paged_attention(q, kv, bt, pos, seg, ("all",), 1.0)
    assert torch.isnan(out).all()


@pytest.mark.parametrize("n,d,e,k", [(50, 5120, 16, 1), (7, 80, 3, 2), (33, 96, 128, 4), (1, 64, 4, 1), (70, 50, 5, 2),
                                     (300, 264, 16, 1)])
def test_moe_route(ops, ref, n, d, e, k):
    h, w = _rand(n, d, seed=1), _rand(e, d, scale=0.05, seed=2)
    ids, gates, logits = ops.moe_route(h, w, k, want_logits=True)
    rid, rg = ref.moe_route(h, w, k)
    assert torch.allclose(logits, h @ w.t(), rtol=1e-4, atol=1e-5)
    assert torch.equal(ids, rid) and torch.allclose(gates, rg, rtol=1e-5, atol=1e-6)


@pytest.mark.parametrize("dt", DT)
@pytest.mark.parametrize("n,d,e,k,delta", [(1, 5120, 16, 1, "experts"), (8, 5120, 16, 1, "experts"), (64, 5120, 128, 1, "plain"),
                                           (1, 5120, 128, 1, "experts"), (64, 5120, 128, 1, "experts"), (256, 5120, 128, 2, "experts"),
                                           (5, 1032, 3, 2, "plain"), (256, 2048, 37, 4, "none"), (3, 8192, 5, 5, "experts")])
def test_norm_and_router_in_one_launch_equal_the_separate_kernels(ops, dt, n, d, e, k, delta):
    """Addition, norm, router logits, choice and grouping fused for steps of few tokens: bit for bit what the norm
    kernel, the logits kernel and the choose-and-group kernel give one after the other."""
    from jax_llm_examples_amd.ops.hip import ExpertSum
    x = _rand(n, d, seed=1)
    w = _rand(d, seed=2) + 1.0
    router = _rand(e, d, scale=0.05, seed=3)
    if delta == "experts":
        m = n * 2
        routed = _rand(m, d, dt=dt, seed=4)
        inv = torch.randperm(m, generator=torch.Generator().manual_seed(5))[: n * 2].to(torch.int32).to(DEV)
        dl = lambda: ExpertSum(routed, inv, 2, _rand(n, d, dt=dt, seed=6), n, d)
    elif delta == "plain":
        dl = lambda: _rand(n, d, dt=dt, seed=4)
    else:
        dl = lambda: None
    x1, x2 = x.clone(), x.clone()
    h_a, h32_a = ops.add_rmsnorm(x1, dl(), w, 1e-5, dt, want32=True)
    ids_a, gates_a, logits_a, group_a = ops.moe_route(h32_a, router, k, want_logits=True, group=True)
    pending = ops.defer_norm(x2, dl(), w, 1e-5, dt)
    calls = []
    inner = ops._call
    ops._call = lambda name, *a: (calls.append(name), inner(name, *a))[1]
    try:
        ids_b, gates_b, logits_b, group_b = ops.moe_route(pending, router, k, want_logits=True, group=True)
    finally:
        ops._call = inner
    assert calls == ["jle_norm_route"], calls
    assert torch.equal(x2, x)  # the residual is not changed in place: its new value is another tensor
    assert torch.equal(pending.residual(), x1) and torch.equal(pending.rows(), h_a)
    assert torch.equal(logits_b, logits_a) and torch.equal(ids_b, ids_a) and torch.equal(gates_b, gates_a)
    for a, b in zip(group_a, group_b):
        assert torch.equal(a, b)
    assert int(ops._tickets.abs().sum()) == 0
    # sizes the fused kernel does not take go through the separate kernels, with the same results
    wide = ops.defer_norm(_rand(2, 520, seed=1), None, None, 1e-5, dt)
    ids_c, _, _ = ops.moe_route(wide, _rand(4, 520, seed=2), 1, group=True)
    assert wide.done and ids_c.shape == (2, 1)


@pytest.mark.parametrize("n,d,e,k", [(700, 320, 16, 1), (600, 90, 6, 2), (520, 64, 37, 3),
                                     # pieces of 4 x 4, 8 x 4 and 8 x 8 (tokens x experts) per wavefront
                                     (2100, 264, 40, 2), (4100, 520, 24, 1), (4099, 136, 70, 3), (2053, 5120, 128, 1)])
def test_router_logits_of_a_token_do_not_depend_on_the_batch(ops, n, d, e, k):
    """Many rows take other kernel shapes than few (larger pieces per wavefront the more rows and experts there
    are); the sums must come out bit for bit the same, or a token's experts would depend on what else is in the
    step."""
    h, w = _rand(n, d, seed=1), _rand(e, d, scale=0.05, seed=2)
    ids, gates, logits = ops.moe_route(h, w, k, want_logits=True)
    # (against the float64 product: a float32 library product is itself off by about as much as the kernel)
    assert torch.allclose(logits.double(), h.double() @ w.double().t(), rtol=1e-4, atol=1e-5)
    for lo, hi in [(0, 1), (n - 1, n), (100, 107), (3, 300)]:
        i2, g2, l2 = ops.moe_route(h[lo:hi].contiguous(), w, k, want_logits=True)
        assert torch.equal(l2, logits[lo:hi]) and torch.equal(i2, ids[lo:hi]) and torch.equal(g2, gates[lo:hi])


@pytest.mark.parametrize("n,d,e,k", [(1, 64, 16, 1), (8, 5120, 16, 1), (64, 96, 128, 2), (1000, 80, 5, 3), (1024, 64, 9, 8),
                                     (1025, 64, 7, 2), (900, 64, 4000, 1), (3000, 72, 16, 1)])
def test_router_and_grouping_in_one_call(ops, n, d, e, k):
    """Few tokens: one block chooses and groups; many tokens, or tables too long for its shared memory: the separate
    kernels.  Either way the same as route, then align."""
    h, w = _rand(n, d, seed=1), _rand(e, d, scale=0.05, seed=2)
    ids, gates, logits = ops.moe_route(h, w, k, want_logits=True)
    ids2, gates2, logits2, grouping = ops.moe_route(h, w, k, want_logits=True, group=True)
    assert torch.equal(ids, ids2) and torch.equal(gates, gates2) and torch.equal(logits, logits2)
    want = ops.moe_align(ids, gates, e, extra_group=True)
    for a, b in zip(want, grouping):
        assert torch.equal(a, b)


def test_moe_route_lowest_index_wins_ties(ops):
    h = _rand(5, 64, seed=1)
    w = _rand(1, 64, seed=2).expand(6, 64).contiguous()  # every expert the same score
    ids, gates = ops.moe_route(h, w, 3)
    assert ids.tolist() == [[0, 1, 2]] * 5


@pytest.mark.parametrize("dt", DT)
@pytest.mark.parametrize("n,d,f,e,k", [(50, 96, 40, 16, 1), (9, 80, 56, 3, 2), (130, 64, 24, 5, 1), (1, 64, 32, 4, 1)])
def test_moe_experts(ops, ref, dt, n, d, f, e, k):
    h = _rand(n, d, dt=dt, seed=1)
    wgu, wd = _rand(e, 2 * f, d, dt=dt, scale=0.2, seed=2), _rand(e, d, f, dt=dt, scale=0.2, seed=3)
    shared = _rand(n, d, dt=dt, seed=4)
    g = torch.Generator().manual_seed(5)
    ids = torch.stack([torch.randperm(e, generator=g)[:k] for _ in range(n)]).to(torch.int32).to(DEV)
    if e > 3:
        ids[ids == 2] = 0  # an expert nobody chose
    gates = torch.rand(n, k, generator=g).to(DEV)
    lazy = ops.moe_experts(h, ids, gates, wgu, wd, shared)  # the pieces; summed by the kernel that uses them
    got = ops.materialize(lazy)
    want = ref.moe_experts(h, ids, gates, wgu, wd, shared)
    assert got.dtype == torch.float32 and lazy.shape == (n, d)
    _assert_close_to_scale(got, want, dt)
    _assert_close_to_scale(ops.materialize(ops.moe_experts(h, ids, gates, wgu, wd, None)),
                           ref.moe_experts(h, ids, gates, wgu, wd, None), dt)
    # residual add + norm reading the pieces = the same on the summed tensor
    x = _rand(n, d, seed=9)
    w = _rand(d, seed=10)
    x1, x2 = x.clone(), x.clone()
    h1, h32 = ops.add_rmsnorm(x1, lazy, w, 1e-5, dt, True)
    h2, h32b = ops.add_rmsnorm(x2, got, w, 1e-5, dt, True)
    assert torch.allclose(x1, x2, rtol=1e-6, atol=1e-6) and torch.allclose(h32, h32b, rtol=1e-5, atol=1e-6)
    x3 = x.clone()
    ops.add_residual(x3, lazy)
    assert torch.allclose(x3, x1, rtol=1e-6, atol=1e-6)
    idx = torch.tensor([n - 1, 0], dtype=torch.int32, device=DEV)
    assert torch.equal(ops.gather_rows(lazy, idx), got[idx.long()])


_SHARED_CASES = [(1, 64, 32, 4, 1), (9, 96, 48, 3, 2), (16, 256, 64, 16, 1), (17, 64, 32, 4, 1), (50, 96, 48, 5, 1)]


# (the streaming layout exists for bfloat16 matrices of whole 16 x 32 tiles only)
@pytest.mark.parametrize("dt,tiled,n,d,f,e,k",
                         [(dt, False, *c) for dt in DT for c in _SHARED_CASES] +
                         [(torch.bfloat16, True, *c) for c in _SHARED_CASES if c[1] % 32 == 0 and c[2] % 32 == 0])
def test_moe_experts_with_the_shared_expert_given_by_its_matrices(ops, ref, dt, tiled, n, d, f, e, k):
    """Up to 16 tokens the shared expert's products go through the routed experts' launches as one more group
    (its matrices stay row-major beside experts in either layout); beyond, through the library.  The same sum."""
    from jax_llm_examples_amd.ops.layout import can_tile, tile_

    h = _rand(n, d, dt=dt, seed=1)
    wgu, wd = _rand(e, 2 * f, d, dt=dt, scale=0.2, seed=2), _rand(e, d, f, dt=dt, scale=0.2, seed=3)
    sgu, sd = _rand(2 * f, d, dt=dt, scale=0.2, seed=4), _rand(d, f, dt=dt, scale=0.2, seed=5)
    g = torch.Generator().manual_seed(5)
    ids = torch.stack([torch.randperm(e, generator=g)[:k] for _ in range(n)]).to(torch.int32).to(DEV)
    gates = torch.rand(n, k, generator=g).to(DEV)
    want = ref.moe_experts(h, ids, gates, wgu, wd, shared_weights=(sgu, sd))
    if tiled:
        assert can_tile(wgu) and can_tile(wd)
        wgu, wd = wgu.clone(), wd.clone()
        tile_(wgu)
        tile_(wd)
    lazy = ops.moe_experts(h, ids, gates, wgu, wd, shared_weights=(sgu, sd), tiled=tiled)
    _assert_close_to_scale(ops.materialize(lazy), want, dt)
    # with the grouping that the router's own call makes (an extra group always), and with one made without
    for extra in (True, False):
        grouping = ops.moe_align(ids, gates, e, extra_group=extra)
        lazy = ops.moe_experts(h, ids, gates, wgu, wd, shared_weights=(sgu, sd), tiled=tiled, grouping=grouping)
        _assert_close_to_scale(ops.materialize(lazy), want, dt)


@pytest.mark.parametrize("n", [1, 8, 64, 2048])
def test_moe_experts_with_128_experts_most_of_them_empty_or_nearly(ops, ref, n):
    """128 experts at serving width (129 groups with the shared expert riding): one token leaves 127 experts
    empty, 2,048 tokens give each about 16 rows and some none (ten experts are never chosen here)."""
    from jax_llm_examples_amd.ops.layout import can_tile, tile_

    dt, d, f, e = torch.bfloat16, 5120, 512, 128
    h = _rand(n, d, dt=dt, seed=1)
    wgu, wd = _rand(e, 2 * f, d, dt=dt, scale=0.02, seed=2), _rand(e, d, f, dt=dt, scale=0.05, seed=3)
    sgu, sd = _rand(2 * f, d, dt=dt, scale=0.02, seed=4), _rand(d, f, dt=dt, scale=0.05, seed=5)
    g = torch.Generator().manual_seed(n)
    ids = (torch.randint(0, e - 10, (n, 1), generator=g) + 5).to(torch.int32).to(DEV)
    gates = torch.rand(n, 1, generator=g).to(DEV)
    want = ref.moe_experts(h, ids, gates, wgu, wd, shared_weights=(sgu, sd))
    assert can_tile(wgu) and can_tile(wd)
    tgu, td = wgu.clone(), wd.clone()
    tile_(tgu)
    tile_(td)
    for tiled, a, b in ((True, tgu, td), (False, wgu, wd)):
        for extra in (True, False):
            grouping = ops.moe_align(ids, gates, e, extra_group=extra)
            lazy = ops.moe_experts(h, ids, gates, a, b, shared_weights=(sgu, sd), tiled=tiled, grouping=grouping)
            _assert_close_to_scale(ops.materialize(lazy), want, dt)
    # the sum that the next norm reads piece by piece
    x = _rand(n, d, seed=7)
    lazy = ops.moe_experts(h, ids, gates, tgu, td, shared_weights=(sgu, sd), tiled=True)
    normed, _ = ops.add_rmsnorm(x.clone(), lazy, None, 1e-5, dt)
    ref_normed, _ = ref.add_rmsnorm(x.clone(), ops.materialize(lazy), None, 1e-5, dt)
    _assert_close_to_scale(normed, ref_normed, dt)


@pytest.mark.parametrize("n,k,e", [(64, 1, 40), (64, 1, 41), (65, 1, 20), (32, 4, 20), (64, 2, 21), (43, 3, 13), (64, 3, 14), (128, 2, 10),
                                   (256, 1, 11), (257, 1, 3), (1, 1, 1)])
def test_moe_align_at_the_edges_of_one_wavefront(ops, n, k, e):
    """As many pairs and experts as one wavefront groups, and one more of either; choices beyond the experts have no row."""
    ids = torch.randint(0, e + 2, (n, k), generator=torch.Generator().manual_seed(n)).int()
    gates = _rand(n, k, seed=5)
    off, tok, gate, inv = (t.cpu() for t in ops.moe_align(ids.to(DEV), gates, e, extra_group=True, note_extra=True))
    flat, order = ids.reshape(-1), [int(r) for r in torch.argsort(ids.reshape(-1), stable=True) if ids.reshape(-1)[r] < e]
    assert off.tolist() == [sum(int(f < i) for f in flat) for i in range(e + 1)] + [len(order) + n]
    assert tok.tolist()[: len(order) + n] == [r // k for r in order] + list(range(n))
    assert torch.equal(gate[: len(order)], gates.cpu().reshape(-1)[order]) and bool((gate[len(order): len(order) + n] == 1).all())
    row = {r: i for i, r in enumerate(order)}
    assert inv.view(n, k + 1).tolist() == [[row.get(t * k + j, -1) for j in range(k)] + [len(order) + t] for t in range(n)]


@pytest.mark.parametrize("n,k,e", [(257, 1, 6), (160, 2, 3), (384, 1, 6), (385, 1, 6), (257, 1, 7), (257, 1, 8), (1024, 1, 63), (1025, 4, 64), (4096, 1, 1), (4097, 1, 300), (8193, 2, 10), (700, 1, 4096), (333, 1, 2048)])
def test_moe_align_of_many_pairs(ops, n, k, e):
    """Runs of pairs that end within 64 and past the ones that a wavefront asks for at once, more experts than a look takes and than
    sixteen wavefronts count; even, all of one expert, and with choices that have no row."""
    g = torch.Generator().manual_seed(n)
    for ids in (torch.randint(0, e + 2, (n, k), generator=g), torch.full((n, k), e - 1), torch.randint(0, min(e, 3), (n, k), generator=g)):
        gates = _rand(n, k, seed=5)
        off, tok, gate, inv = (t.cpu() for t in ops.moe_align(ids.int().to(DEV), gates, e, extra_group=True, note_extra=True))
        flat = ids.reshape(-1)
        order = torch.argsort(flat, stable=True)
        order = order[flat[order] < e]
        rows = order.numel()
        assert torch.equal(off[: e + 1].long(), torch.cat([torch.zeros(1), torch.bincount(flat[flat < e], minlength=e)]).cumsum(0).long())
        assert off[e + 1] == rows + n and torch.equal(tok[: rows + n].long(), torch.cat([order // k, torch.arange(n)]))
        assert torch.equal(gate[:rows], gates.cpu().reshape(-1)[order])
        want = torch.full((n * k,), -1)
        want[order] = torch.arange(rows)
        assert torch.equal(inv.view(n, k + 1).long(), torch.cat([want.view(n, k), rows + torch.arange(n)[:, None]], 1))


def test_moe_align_is_a_stable_grouping(ops):
    g = torch.Generator().manual_seed(0)
    ids = torch.randint(0, 7, (300, 2), generator=g).to(torch.int32).to(DEV)
    gates = torch.rand(300, 2, generator=g).to(DEV)
    off, tok, gate, inv = ops.moe_align(ids, gates, 7)
    flat = ids.flatten().cpu()
    off, tok, gate, inv = off.cpu(), tok.cpu(), gate.cpu(), inv.cpu()
    assert off[0] == 0 and off[-1] == 600
    for e in range(7):
        rows = (flat == e).nonzero().squeeze(-1)
        assert off[e + 1] - off[e] == rows.numel()
        assert torch.equal(inv[rows], torch.arange(int(off[e]), int(off[e + 1]), dtype=torch.int32))  # in order
        assert torch.equal(tok[off[e]: off[e + 1]], (rows // 2).to(torch.int32))
    assert torch.equal(gate[inv.long()], gates.flatten().cpu())
    # one more group that holds every token once
    off2, tok2, gate2, inv2 = (t.cpu() for t in ops.moe_align(ids, gates, 7, extra_group=True))
    assert torch.equal(off2[:8], off) and off2[8] == 900 and torch.equal(inv2, inv)
    assert torch.equal(tok2[:600], tok) and torch.equal(tok2[600:], torch.arange(300, dtype=torch.int32))
    assert torch.equal(gate2[:600], gate) and torch.equal(gate2[600:], torch.ones(300))


@pytest.mark.parametrize("dt", DT)
def test_product_kernel_and_lm_head(ops, ref, dt):
    a, b = _rand(33, 52, dt=dt, seed=1), _rand(70, 52, dt=dt, seed=2)
    _assert_close_to_scale(ops.gemm(a, b), ref.linear(a, b), dt)
    gu = _rand(2 * 24, 52, dt=dt, seed=6)
    for rows in (33, 100):  # few rows (weight streaming in bfloat16) and many
        aa = _rand(rows, 52, dt=dt, seed=7)
        _assert_close_to_scale(ops.swiglu_linear(aa, gu), ref.swiglu_linear(aa, gu), dt)
        _assert_close_to_scale(ops.linear(aa, b), ref.linear(aa, b), dt)
    h, w = _rand(5, 80, dt=dt, seed=3), _rand(311, 80, dt=dt, seed=4)
    got = ops.lm_head(h, w)
    assert got.dtype == torch.float32 and got.shape == (5, 311)
    assert torch.allclose(got, ref.lm_head(h, w), rtol=2e-5, atol=2e-5)  # float32 accumulation and output
    _assert_close_to_scale(ops.linear(h, w), ref.linear(h, w), dt)


def test_float32_products_are_true_float32(ops):
    # a reduced-precision matrix mode (tf32/xf32: 10 mantissa bits) would lose the small term
    a = torch.tensor([[1.0, 2.0 ** -14]], device=DEV).repeat(4, 64)  # 128 columns
    b = torch.ones(8, 128, device=DEV)
    want = 64 * (1.0 + 2.0 ** -14)
    for out in (ops.linear(a, b), ops.lm_head(a, b), ops.gemm(a, b)):
        assert torch.allclose(out, torch.full_like(out, want), rtol=1e-7)


@pytest.mark.parametrize("rows", [1, 64, 2048])
@pytest.mark.parametrize("k", [5120, 8192, 16384])
def test_float32_products_are_true_float32_at_serving_sizes(ops, rows, k):
    """The shapes the dense projections really have (which algorithm a library picks depends on them), against
    a float64 product.  Rows of 1 + 2^-12, -1, 1 + 2^-12, -1, ... times ones: every partial sum over neighbouring
    terms is exact in float32 in whatever order it is taken, and the result is k / 2 * 2^-12; a mode that keeps
    10 mantissa bits of the operands gives 0.  And random operands against the float64 product."""
    nout = 384
    a = torch.tensor([[1.0 + 2.0 ** -12, -1.0]], device=DEV).repeat(rows, k // 2)
    b = torch.ones(nout, k, device=DEV)
    exact = k / 2 * 2.0 ** -12
    ar, br = _rand(rows, k, seed=11), _rand(nout, k, seed=12)
    want = (ar.double() @ br.double().t())
    scale = (ar.double().abs() @ br.double().abs().t())
    for name, fn in (("linear", ops.linear), ("lm_head", ops.lm_head), ("gemm", ops.gemm)):
        out = fn(a, b)
        assert float((out.double() - exact).abs().max()) <= 1e-6 * exact, name
        err = float(((fn(ar, br).double() - want).abs() / scale).max())
        assert err < 2e-6, f"{name}: {err:.3g} of the sum of the terms' sizes"


@pytest.mark.parametrize("rows,nout,k", [(1, 2, 4), (2, 513, 1000), (3, 64, 36), (4, 1030, 2044), (5, 6, 256), (8, 70, 1284),
                                         (128, 2056, 4096), (512, 4096, 4096), (300, 136, 256), (1, 8, 32), (257, 264, 8224)])
def test_dense_float32_products(ops, rows, nout, k):
    """The kernels for up to eight rows and for many (tiles of 128 x 128, stages of 32 k, ranges of k), and with the
    activation.  A sum of K products carries at most a rounding of 2^-24 of the terms' sizes per addition that follows
    one; the kernel for few rows adds up K / 256 numbers and 30 more a number, the one in parts rounds 192
    times at most in a stage of 32, then once a stage, and leaves out at most 2^-24 of a product."""
    x, w = _rand(rows, k, seed=21), _rand(nout, k, seed=22)
    want, size = x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t()
    gate, up = want.chunk(2, -1) if nout % 2 == 0 else (None, None)
    kernels = [(ops.gemm_f32_rows, k / 256 * 4 + 40, 0.0)] if rows <= 8 else []
    if k % 32 == 0 and nout % 8 == 0:
        kernels.append((ops.gemm_f32_split, k / 32 + 200, 2.0 ** -24))
        kernels.append((lambda *a: ops.gemm_f32_split(*a, ranges=1 if len(a) > 2 else min(7, k // 32)), k / 32 + 200, 2.0 ** -24))
    for fn, adds, left in kernels:
        bound = size * (adds * 2.0 ** -24 + left)
        assert bool(((fn(x, w).double() - want).abs() <= bound).all())
        if gate is not None:
            # (|silu'| and |gelu'| < 1.13; what the kernel's own form of either adds is float32 roundings)
            for act, f in ((0, torch.nn.functional.silu(gate)), (1, torch.nn.functional.gelu(gate, approximate="tanh"))):
                b = 1.13 * bound[:, :nout // 2] * up.abs() + (f.abs() + 2.0 ** -19 * gate.abs()) * bound[:, nout // 2:]
                got = fn(x, w, act).double()
                assert bool(((got - f * up).abs() <= 1.01 * b + 2.0 ** -19 * (gate * up).abs() + 1e-30).all()), act
    ranges = ops.split_ranges(rows, nout, k, False, ops._compute_units)
    assert ranges or (rows, nout, k) != (512, 4096, 4096)
    if rows <= 4 or ranges:  # (where the way leads here)
        assert torch.equal(ops.linear(x, w), ops.gemm_f32_split(x, w, -1, ranges) if ranges else ops.gemm_f32_rows(x, w))


@pytest.mark.parametrize("rows,nout,k", [(9, 2, 4), (16, 64, 64), (17, 130, 36), (33, 1000, 516), (64, 1024, 1024), (128, 512, 2048), (32, 2048, 2048),
                                         (127, 62, 2044), (48, 2048, 300)])
def test_dense_float32_products_of_tens_of_rows(ops, rows, nout, k):
    """The experts' kernel for few rows with one group, the way the dense products of such sizes go.  A wavefront adds up every
    eighth chunk of 32 k, the instruction four at a time: k / 32 + 40 roundings at most."""
    x, w = _rand(rows, k, seed=41), _rand(nout, k, seed=42)
    want, size = x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t()
    bound = size * (k / 32 + 40) * 2.0 ** -24
    got = ops.gemm_f32_skinny(x, w)
    assert bool(((got.double() - want).abs() <= bound).all())
    assert torch.equal(got, ops.linear(x, w)) or not ops.f32_tiles_pay(rows, nout, k, False)
    gate, up = want.chunk(2, -1)
    got = ops.gemm_f32_skinny(x, w, swiglu=True)
    assert torch.equal(got, ops.swiglu_linear(x, w)) or not ops.f32_tiles_pay(rows, nout, k, True)
    b = 1.13 * bound[:, :nout // 2] * up.abs() + (gate.abs() + 2.0 ** -19 * gate.abs()) * bound[:, nout // 2:]
    assert bool(((got.double() - torch.nn.functional.silu(gate) * up).abs() <= 1.01 * b + 2.0 ** -19 * (gate * up).abs() + 1e-30).all())
    gelu = ops.swiglu_linear(x, w, "gelu_tanh").double()  # (has no kernel here: the library's and a pass of its own)
    assert float((gelu - torch.nn.functional.gelu(gate, approximate="tanh") * up).norm() / gelu.norm()) < 1e-5


@pytest.mark.parametrize("k", [32, 256, 2080, 8192])
def test_dense_float32_products_in_parts_lose_no_part(ops, k):
    """The product of operands in three bfloat16 parts each is a float32 product: of sums of like terms, of a single
    term, and with the leading parts cancelled so that each of the six partial products is all that is left."""
    x, w = _rand(130, k, seed=31), _rand(136, k, seed=32)
    want = x.double() @ w.double().t()
    # a rounding of the whole per stage of 32 k and a few beside; one partial product left out alone is 2e-6
    assert float((ops.gemm_f32_split(x, w).double() - want).norm() / want.norm()) < 2.0 ** -24 * (k / 32 + 4) ** 0.5
    one = torch.arange(k, device=DEV)[None] == (torch.arange(130, device=DEV) % k)[:, None]
    for ranges in (1, min(3, k // 32)):
        want = torch.where(one, x, 0.0).double() @ w.double().t()
        got = ops.gemm_f32_split(torch.where(one, x, 0.0), w, -1, ranges).double()
        # left out 2^-24 at most, the sum of what is kept rounded once (and its small terms a little)
        assert float(((got - want).abs() / want.abs()).max()) < 1.02 * 2.0 ** -23
    m, l = 2.0 ** -9, 2.0 ** -18  # 1 + m + l: its three parts
    for a, b, less in ((1 + m + l, 1.0, 1.0), (1.0, 1 + m + l, 1.0), (1 + l, 1.0, 1.0), (1.0, 1 + l, 1.0),
                       (1 + m, 1 + m, 1 + 2 * m), (1 + 2.0 ** -23, 1.0, 1.0), (1.0, 1 + 2.0 ** -23, 1.0)):
        x, w = torch.zeros(4, k, device=DEV), torch.zeros(8, k, device=DEV)
        x[:, 5], w[:, 5], x[:, 17], w[:, 17] = a, b, -less, 1.0
        assert torch.equal(ops.gemm_f32_split(x, w), torch.full((4, 8), a * b - less, device=DEV)), (a, b, less)


def test_dense_float32_products_of_small_numbers_beside_large_ones(ops):
    """Numbers whose parts are too small for bfloat16, in rows that hold large ones (which meet a zero), and products whose
    partial products are too small: what float32 holds is not lost.  Rows of zeros stay zeros."""
    x, w = _rand(132, 320, seed=35) * 1e-36, _rand(136, 320, seed=36) * 1e12
    x[:, 3], w[:, 3] = 1.0, 0.0
    x[70] = 0.0
    y, v = _rand(132, 320, seed=37) * 2.0 ** -59, _rand(136, 320, seed=38) * 2.0 ** -59
    for a, b in ((x, w), (w, x), (y, v)):
        want, size = a.double() @ b.double().t(), a.double().abs() @ b.double().abs().t()
        for ranges in (1, 4):
            got = ops.gemm_f32_split(a, b, -1, ranges).double()
            assert bool(((got - want).abs() <= size * (320 / 4 + 40) * 2.0 ** -24).all())  # (a rounding per float32 sum of 4)


@pytest.mark.parametrize("act", [0, 1])
def test_dense_float32_products_of_special_numbers_with_the_activation(ops, act):
    """Infinities and NaN in some rows of either operand, and rows of very small numbers, behind the fused activation."""
    x, w = _rand(200, 320, seed=33), _rand(272, 320, seed=34, scale=0.1)
    x[3, 7], x[190, 9] = float("inf"), float("nan")
    w[135, 0], w[140, 100] = -float("inf"), float("nan")
    x[50] *= 1e-36
    gate, up = (x.double() @ w.double().t()).float().double().chunk(2, -1)
    f = torch.nn.functional.silu if act == 0 else lambda z: torch.nn.functional.gelu(z, approximate="tanh")
    want, got = f(gate) * up, ops.gemm_f32_split(x, w, act).double()
    # (silu as the kernels form it: -inf / inf is NaN)
    ok = torch.isfinite(want) & ~((gate / (1 + torch.exp(-gate)) * up).isnan() if act == 0 else want.isnan())
    assert bool(torch.isfinite(got[ok]).all()) and not bool(torch.isfinite(got[~ok]).any())
    size = x.double().abs() @ w.double().abs().t()
    size = torch.where(torch.isfinite(size), size, 0.0)
    s_gate, s_up = size.chunk(2, -1)
    # each sum as in test_dense_float32_products; |f'| < 1.13, f itself to a few roundings
    e_gate, e_up = ((320 / 32 + 200) * 2.0 ** -24 * s for s in (s_gate, s_up))
    bound = 1.13 * e_gate * up.abs() + (f(gate).abs() + 2.0 ** -19 * gate.abs()) * e_up + 2.0 ** -19 * (gate * up).abs()
    assert bool(((got - want).abs()[ok] <= 1.01 * bound[ok] + 1e-44).all())


def test_dense_float32_products_of_special_numbers(ops):
    """Infinities, NaN and numbers beyond bfloat16's largest give what float32 gives; rows of very small numbers
    lose nothing."""
    x, w = _rand(200, 320, seed=23), _rand(136, 320, seed=24)
    x[3, 7], x[190, 9], x[70, 5], x[131, 319] = float("inf"), float("nan"), 3.4e38, -float("inf")
    w[135, 0], w[5, 100] = -float("inf"), 3.4e38
    x[40] = 0.0
    want = (x.cpu().double() @ w.cpu().double().t()).float()
    got = ops.gemm_f32_split(x, w).cpu()
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf())
    assert torch.equal(got[got.isinf()], want[want.isinf()])
    x, w = _rand(130, 320, seed=25) * 1e-36, _rand(136, 320, seed=26) * 1e12
    want, size = x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t()
    assert bool(((ops.gemm_f32_split(x, w).double() - want).abs() <= size * (320 / 4 + 40) * 2.0 ** -24).all())


@pytest.mark.parametrize("n,d,f,e,k", [(1, 64, 32, 4, 1), (8, 5120, 96, 16, 1), (64, 260, 36, 128, 2), (100, 128, 64, 5, 1),
                                       (128, 512, 256, 16, 1), (50, 1028, 44, 3, 2), (129, 64, 16, 1, 1)])
def test_float32_grouped_product_on_the_float32_matrix_instructions(ops, n, d, f, e, k):
    """The weight-streaming float32 product (gemm_f32.hip) against float64: grouped, gathered, scaled, with and
    without the fused activation; sizes that leave partial tiles, chunks and groups without rows."""
    h = _rand(n, d, seed=1)
    wgu, wd = _rand(e, 2 * f, d, scale=0.1, seed=2), _rand(e, d, f, scale=0.1, seed=3)
    g = torch.Generator().manual_seed(n)
    ids = torch.stack([torch.randperm(e, generator=g)[:k] for _ in range(n)]).to(torch.int32).to(DEV)
    if e > 2:
        ids[ids == 1] = 2  # a group without rows
    gates = torch.rand(n, k, generator=g).to(DEV)
    off, tok, gate, inv = ops.moe_align(ids, gates, e)
    act = ops.gemm_f32_skinny(h, wgu, offsets=off, a_rows=tok, scale=gate, swiglu=True)
    gu = ops.gemm_f32_skinny(h, wgu, offsets=off, a_rows=tok, scale=gate)
    sorted_ids = ids.flatten()[torch.argsort(inv.long())].long()
    x64 = h.double()[tok.long()] * gate.double()[:, None]
    want_gu = torch.einsum("nk,nok->no", x64, wgu.double()[sorted_ids])
    want_act = torch.nn.functional.silu(want_gu[:, :f]) * want_gu[:, f:]
    assert float((gu.double() - want_gu).abs().max() / want_gu.abs().max()) <= 3e-6
    assert float((act.double() - want_act).abs().max() / want_act.abs().max()) <= 3e-6
    out = ops.gemm_f32_skinny(act, wd, offsets=off)
    want = torch.einsum("nk,nok->no", act.double(), wd.double()[sorted_ids])
    assert float((out.double() - want).abs().max() / want.abs().max()) <= 3e-6
    # one group without offsets, and the result of a row does not depend on what else is in the launch
    dense = ops.gemm_f32_skinny(h, wgu[0])
    assert float((dense.double() - h.double() @ wgu[0].double().t()).abs().max() / dense.abs().max()) <= 3e-6
    assert torch.equal(ops.gemm_f32_skinny(h[:1].contiguous(), wgu[0]), dense[:1])
    with pytest.raises(Exception, match="multiple of 4"):
        ops.gemm_f32_skinny(h[:, : d - 2].contiguous(), wgu[:, :, : d - 2].contiguous())


@pytest.mark.parametrize("n,d,f,e,k", [(1, 64, 64, 4, 1), (50, 128, 64, 4, 1), (300, 192, 128, 3, 2), (700, 64, 192, 5, 1),
                                       (450, 320, 64, 2, 1), (2100, 5120, 128, 16, 1), (200, 1088, 448, 128, 2)])
def test_float32_grouped_product_for_many_rows_on_the_float32_matrix_instructions(ops, n, d, f, e, k):
    """The float32 product whose wavefronts hold up to 192 rows of a group (gemm_f32.hip) against float64: grouped,
    gathered, scaled, with and without the fused activation; groups of more than 192 rows (several passes), of a
    few rows and of none, rows that fill no tile."""
    h = _rand(n, d, seed=1)
    wgu, wd = _rand(e, 2 * f, d, scale=0.1, seed=2), _rand(e, d, f, scale=0.1, seed=3)
    g = torch.Generator().manual_seed(n)
    ids = torch.stack([torch.randperm(e, generator=g)[:k] for _ in range(n)]).to(torch.int32).to(DEV)
    if e > 2:
        ids[ids == 1] = 2  # a group without rows, and one with twice its share
    gates = torch.rand(n, k, generator=g).to(DEV)
    off, tok, gate, inv = ops.moe_align(ids, gates, e)
    act = ops.gemm_f32_stream(h, wgu, offsets=off, a_rows=tok, scale=gate, swiglu=True)
    gu = ops.gemm_f32_stream(h, wgu, offsets=off, a_rows=tok, scale=gate)
    sorted_ids = ids.flatten()[torch.argsort(inv.long())].long()
    x64 = h.double()[tok.long()] * gate.double()[:, None]
    want_gu = torch.empty(tok.numel(), 2 * f, dtype=torch.float64, device=DEV)
    for j in range(e):
        rows = sorted_ids == j
        want_gu[rows] = x64[rows] @ wgu[j].double().t()
    want_act = torch.nn.functional.silu(want_gu[:, :f]) * want_gu[:, f:]
    assert float((gu.double() - want_gu).abs().max() / want_gu.abs().max()) <= 3e-6
    assert float((act.double() - want_act).abs().max() / want_act.abs().max()) <= 3e-6
    out = ops.gemm_f32_stream(act, wd, offsets=off)
    want = torch.empty(tok.numel(), d, dtype=torch.float64, device=DEV)
    for j in range(e):
        rows = sorted_ids == j
        want[rows] = act.double()[rows] @ wd[j].double().t()
    assert float((out.double() - want).abs().max() / want.abs().max()) <= 3e-6
    # one group without offsets, and the result of a row does not depend on what else is in the launch
    # (measured against the sum of the terms' sizes, as for the dense projections above: the sums over 5,120 terms
    # are formed one stage after the other)
    dense = ops.gemm_f32_stream(h, wgu[0])
    terms = h.double().abs() @ wgu[0].double().abs().t()
    assert float(((dense.double() - h.double() @ wgu[0].double().t()).abs() / terms).max()) < 2e-6
    assert torch.equal(ops.gemm_f32_stream(h[:1].contiguous(), wgu[0]), dense[:1])
    with pytest.raises(Exception, match="multiple of 64"):
        ops.gemm_f32_stream(h[:, : d - 32].contiguous(), wgu[:, :, : d - 32].contiguous())
    # through the experts' entry: more rows than the few-rows kernel takes
    if n * k > ops.F32_SKINNY_ROWS:
        calls = []
        inner = ops._call
        ops._call = lambda name, *a: (calls.append(name), inner(name, *a))[1]
        try:
            got = ops.materialize(ops.moe_experts(h, ids, gates, wgu, wd, None))
        finally:
            ops._call = inner
        assert calls.count("jle_gemm_f32_stream") == 2, calls
        want_sum = torch.zeros(n, d, dtype=torch.float64, device=DEV)
        want_sum.index_add_(0, tok.long(), want)
        assert float((got.double() - want_sum).abs().max() / want_sum.abs().max()) <= 3e-6


def test_sampling(ops, ref):
    g = torch.Generator().manual_seed(0)
    V = 1000
    logits = torch.randn(6, V, generator=g).to(DEV)
    logits[0, 17] = logits[0, 400] = 9.0  # two equal maxima: the lower id
    z = torch.zeros(6, dtype=torch.int32, device=DEV)
    greedy = ops.sample(logits, torch.zeros(6, device=DEV), z, z, z)
    assert greedy.tolist() == torch.argmax(logits, -1).tolist() and greedy[0] == 17
    temp = torch.tensor([0.0, 0.7, 1.0, 1.3, 1.0, 1.0], device=DEV)
    topk = torch.tensor([0, 0, 5, 16, 1, 0], dtype=torch.int32, device=DEV)
    seeds = torch.tensor([1, 2, 3, 4, 5, 6], dtype=torch.int32, device=DEV)
    for c in range(4):
        ctr = torch.full((6,), c, dtype=torch.int32, device=DEV)
        got = ops.sample(logits, temp, topk, seeds, ctr)
        want = ref.sample(logits.cpu(), temp.cpu(), topk.cpu(), seeds.cpu(), ctr.cpu())
        assert got.tolist() == want.tolist()
        assert got[4] == torch.argmax(logits[4])  # top_k = 1 is greedy
        assert int(got[2]) in torch.topk(logits[2], 5).indices.tolist()
    # a request's draw does not depend on what else is in the batch
    alone = ops.sample(logits[3:4].contiguous(), temp[3:4].contiguous(), topk[3:4].contiguous(),
                       seeds[3:4].contiguous(), torch.tensor([2], dtype=torch.int32, device=DEV))
    ctr = torch.full((6,), 2, dtype=torch.int32, device=DEV)
    assert alone[0] == ops.sample(logits, temp, topk, seeds, ctr)[3]


def test_sampling_frequencies_follow_softmax(ops):
    p = torch.tensor([0.5, 0.25, 0.15, 0.07, 0.03])
    n = 4000
    logits = torch.log(p)[None].repeat(n, 1).to(DEV) * 2.0  # temperature 2 undoes the factor
    out = ops.sample(logits, torch.full((n,), 2.0, device=DEV), torch.zeros(n, dtype=torch.int32, device=DEV),
                     torch.arange(n, dtype=torch.int32, device=DEV), torch.zeros(n, dtype=torch.int32, device=DEV))
    freq = torch.bincount(out.cpu().long(), minlength=5).float() / n
    sigma = torch.sqrt(p * (1 - p) / n)
    assert ((freq - p).abs() < 4 * sigma).all(), (freq, p)


@pytest.mark.parametrize("m,nout,k", [(1, 64, 64), (8, 70, 104), (16, 33, 32), (17, 96, 40), (40, 500, 264),
                                       (64, 130, 5120), (5, 1000, 8192), (3, 80, 1096)])
@pytest.mark.parametrize("out_f32", [False, True])
def test_weight_streaming_product(ops, ref, m, nout, k, out_f32):
    a, b = _rand(m, k, dt=torch.bfloat16, seed=1), _rand(nout, k, dt=torch.bfloat16, scale=0.1, seed=2)
    got = ops.gemm_skinny(a, b, out_f32=out_f32)
    want = a.float() @ b.float().t()
    assert got.dtype == (torch.float32 if out_f32 else torch.bfloat16)
    err = float((got.float() - want).abs().max() / want.abs().max())
    assert err <= (2e-5 if out_f32 else 5e-3), err  # float32 out: only the order of the sum differs


@pytest.mark.parametrize("m", [1, 8, 16])
@pytest.mark.parametrize("nout,k", [(5120, 320), (5120, 8192), (1024, 264), (9216, 5120), (2048, 512)])
def test_weight_streaming_product_with_row_tiles_cut_along_k(ops, m, nout, k):
    """Row tiles that do not fill a round of the compute units are cut along K, each slice a block of its own,
    and the slices' sums are added by the tile's last block in the slices' order: the same bits every time, in
    both layouts, and the tickets are back at zero."""
    from jax_llm_examples_amd.ops.layout import can_tile, tile_
    tiles = -(-nout // 16)
    cut, slices = ops._k_slices(tiles)
    assert cut > 0 and (cut * slices) % ops._compute_units == 0, "sizes chosen so that tiles are cut"
    a, b = _rand(m, k, dt=torch.bfloat16, seed=1), _rand(nout, k, dt=torch.bfloat16, scale=0.1, seed=2)
    want = a.float() @ b.float().t()
    got = ops.gemm_skinny(a, b, out_f32=True)
    assert float((got - want).abs().max() / want.abs().max()) <= 2e-5
    whole = ops.gemm_skinny(a, b, out_f32=True, balance=False)  # (sums in another order: other blocks, other bits)
    assert float((whole - want).abs().max() / want.abs().max()) <= 2e-5
    for _ in range(3):
        assert torch.equal(ops.gemm_skinny(a, b, out_f32=True), got)
    if can_tile(b):
        bt = b.clone()
        tile_(bt)
        assert torch.equal(ops.gemm_skinny(a, bt, out_f32=True, tiled=True), got)
    assert int(ops._slice_tickets.abs().sum()) == 0


@pytest.mark.parametrize("n,e,nout,k", [(1, 16, 5120, 512), (2, 128, 5120, 256), (8, 16, 5120, 8192), (7, 128, 320, 64),
                                        (16, 40, 2048, 128)])
def test_weight_streaming_product_over_group_slots(ops, n, e, nout, k):
    """A grouped product of few rows is launched over as many group slots as it has rows (slot j: the j-th group
    that has rows), with a last group whose matrix is a tensor of its own: the same result as over every group."""
    dt = torch.bfloat16
    g = torch.Generator().manual_seed(n)
    ids = torch.randint(0, e, (n, 1), generator=g).to(torch.int32).to(DEV)
    gates = torch.rand(n, 1, generator=g).to(DEV)
    off, tok, gate, inv = ops.moe_align(ids, gates, e, extra_group=True)
    x = _rand(2 * n, k, dt=dt, seed=1)  # (rows already grouped: the second product of an expert layer)
    w, w_last = _rand(e, nout, k, dt=dt, scale=0.1, seed=2), _rand(nout, k, dt=dt, scale=0.1, seed=3)
    got = ops.gemm_skinny(x, w, offsets=off, b_last=w_last, out_f32=True)
    every = ops.gemm_skinny(x, w, offsets=off, b_last=w_last, out_f32=True, balance=False)
    sorted_ids = ids.flatten()[tok[:n].long()].long()
    want = torch.cat([torch.einsum("nk,nok->no", x[:n].float(), w[sorted_ids].float()),
                      x[n:].float() @ w_last.float().t()])
    assert float((got - want).abs().max() / want.abs().max()) <= 2e-5
    assert float((every - want).abs().max() / want.abs().max()) <= 2e-5
    # (tiles are cut only in launches of one or two group slots; with no tile cut the same blocks form the same sums)
    if ops._k_slices(-(-nout // 16))[0] == 0 or 2 * n > ops.CUT_SLOTS:
        assert torch.equal(got, every)
    # gathered rows, scaled, with the fused activation (the first product of an expert layer)
    h = _rand(n, k, dt=dt, seed=4)
    wgu, wgu_last = _rand(e, 2 * 64, k, dt=dt, scale=0.1, seed=5), _rand(2 * 64, k, dt=dt, scale=0.1, seed=6)
    a1 = ops.gemm_skinny(h, wgu, offsets=off, a_rows=tok, scale=gate, swiglu=True, b_last=wgu_last, rows=2 * n)
    a2 = ops.gemm_skinny(h, wgu, offsets=off, a_rows=tok, scale=gate, swiglu=True, b_last=wgu_last, rows=2 * n,
                         balance=False)
    assert torch.equal(a1, a2)
    assert int(ops._slice_tickets.abs().sum()) == 0


@pytest.mark.parametrize("n,d,f,e,k", [(8, 128, 48, 16, 1), (64, 5120, 64, 16, 1), (20, 264, 40, 3, 2), (3, 64, 24, 128, 1)])
def test_weight_streaming_product_grouped_with_swiglu(ops, ref, n, d, f, e, k):
    dt = torch.bfloat16
    h = _rand(n, d, dt=dt, seed=1)
    wgu = _rand(e, 2 * f, d, dt=dt, scale=0.1, seed=2)
    g = torch.Generator().manual_seed(5)
    ids = torch.stack([torch.randperm(e, generator=g)[:k] for _ in range(n)]).to(torch.int32).to(DEV)
    if n == 64:
        ids[:40] = 3  # one expert with more rows than one tile of 16
    gates = torch.rand(n, k, generator=g).to(DEV)
    off, tok, gate, inv = ops.moe_align(ids, gates, e)
    act = ops.gemm_skinny(h, wgu, offsets=off, a_rows=tok, scale=gate, swiglu=True)
    gu = ops.gemm(h, wgu, offsets=off, a_rows=tok, scale=gate, out_f32=True)  # the general kernel, float32 result
    want = torch.nn.functional.silu(gu[:, :f]) * gu[:, f:]
    assert act.shape == (n * k, f)
    assert float((act.float() - want).abs().max() / want.abs().max()) <= 5e-3
    plain = ops.gemm_skinny(h, wgu, offsets=off, a_rows=tok, scale=gate, out_f32=True)
    assert float((plain - gu).abs().max() / gu.abs().max()) <= 2e-5


@pytest.mark.parametrize("tiled", [False, True])
@pytest.mark.parametrize("counts,nout,k", [([17, 0, 32, 33, 1], 96, 160), ([24], 4096 * 16, 64), ([40, 8], 80, 72),
                                           ([16, 15, 64, 9], 8192, 96), ([40, 8] * 180, 80, 72),
                                           ([17, 0, 32, 33, 1] * 70, 96, 160)])
def test_weight_streaming_product_of_fuller_groups(ops, counts, nout, k, tiled):
    """Groups of eight rows and more on average take 32 rows a block where the row tiles fill the card, and with many rows
    of W two row tiles: groups that end at, before and behind 16 and 32 rows, empty ones between."""
    if tiled and (k % 32 or nout % 32):
        pytest.skip("no whole tiles")
    m, e = sum(counts), len(counts)
    x, w = _rand(m, k, dt=torch.bfloat16, seed=1), _rand(e, nout, k, dt=torch.bfloat16, scale=0.1, seed=2)
    off = torch.tensor([0] + counts).cumsum(0).int().to(DEV)
    stored = w
    if tiled:
        from jax_llm_examples_amd.ops.layout import tile_
        stored = w.clone()
        tile_(stored)
    got = ops.gemm_skinny(x, stored, offsets=off, out_f32=True, tiled=tiled)
    act = ops.gemm_skinny(x, stored, offsets=off, swiglu=True, tiled=tiled)
    o = 0
    for c, we in zip(counts, w):
        want = x[o: o + c].double() @ we.double().T
        if c:
            # float32 sums of k products of bfloat16 numbers: sqrt(k) 2^-24 of the terms' size, with room
            assert float((got[o: o + c].double() - want).norm() / want.norm()) <= 2e-6
            want = torch.nn.functional.silu(want[:, : nout // 2]) * want[:, nout // 2:]
            assert float((act[o: o + c].double() - want).norm() / want.norm()) <= 2.0 ** -8  # (rounded to bfloat16)
        o += c


@pytest.mark.parametrize("counts,nout,k,swiglu", [
    ([1, 0, 31, 32, 33, 64, 65], 96, 256, False),           # few rows, whole rounds of stages only at the end
    ([128, 129, 160, 161, 192, 193], 528, 512, False),      # every number of row tiles; a second block of W of one tile
    ([224, 225, 256, 257, 512, 513, 700], 544, 768, True),  # one, two and three tiles of rows; gate and up
    ([3, 0, 280] * 50, 64, 256, False),                     # more groups than a look takes
    ([256], 2304, 256, True),                               # more than eight blocks of W
    # every number of row tiles and one row more, full tiles among them, over twelve stages: every ring goes round more than once
    ([1, 32, 64, 65, 96, 97, 128, 129, 160, 161, 192, 193, 224, 225, 256, 257, 512], 288, 768, False),
    ([1, 32, 64, 65, 96, 97, 128, 129, 160, 161, 192, 193, 224, 225, 256, 257, 512], 288, 768, True)])
def test_wide_tiles_of_the_weight_streaming_product(ops, monkeypatch, counts, nout, k, swiglu):
    """The kernel for many rows a group gives the bits of the one that takes them in passes (the same sums in the same
    order), with the rows gathered and scaled; that one is tested against the general product elsewhere."""
    from jax_llm_examples_amd.ops.layout import tile_
    m, e = sum(counts), len(counts)
    x, w = _rand(m + 3, k, dt=torch.bfloat16, seed=1), _rand(e, nout, k, dt=torch.bfloat16, scale=0.1, seed=2)
    tile_(w)
    off = torch.tensor([0] + counts).cumsum(0).int().to(DEV)
    rows = torch.randperm(m + 3, generator=torch.Generator().manual_seed(3))[:m].int().to(DEV)
    scale = _rand(m, seed=4)
    got = []
    monkeypatch.setattr(ops, "stream_half", lambda *a: False)
    for wide in (False, True):
        monkeypatch.setattr(ops, "stream_wide", lambda *a, wide=wide: wide)
        got.append(ops.gemm_stream(x, w, offsets=off, a_rows=rows, scale=scale, swiglu=swiglu, rows=m))
    assert torch.equal(*got)


@pytest.mark.parametrize("counts,nout,k", [
    ([1, 0, 32, 33, 64, 65, 96, 97, 128, 129], 128, 256),        # every number of row tiles
    ([160, 161, 192, 193, 224, 225, 256, 257], 144, 512),        # a second block of W of one tile
    ([288, 0, 289, 576, 577, 900], 1168, 256),                   # the most rows of a tile and one more; more than eight blocks of W
    ([1, 32, 64, 65, 96, 97, 128, 129, 160, 161, 192, 193, 224, 225, 256, 257, 288, 289, 576], 144, 768)])  # twelve stages
def test_narrower_wide_tiles_of_the_weight_streaming_product(ops, monkeypatch, counts, nout, k):
    """The bits of the kernel that takes the rows in passes, rows gathered and scaled; rows that no group has are left alone."""
    from jax_llm_examples_amd.ops.layout import tile_
    m, e = sum(counts), len(counts)
    x, w = _rand(m + 3, k, dt=torch.bfloat16, seed=1), _rand(e, nout, k, dt=torch.bfloat16, scale=0.1, seed=2)
    tile_(w)
    off = torch.tensor([0] + counts).cumsum(0).int().to(DEV)
    rows = torch.randperm(m + 3, generator=torch.Generator().manual_seed(3)).int().to(DEV)
    scale = _rand(m + 3, seed=4)
    got = []
    monkeypatch.setattr(ops, "stream_wide", lambda *a: False)
    monkeypatch.setattr(ops, "stream_cuts", lambda *a: (0, 1))
    for half in (False, True):
        monkeypatch.setattr(ops, "stream_half", lambda *a, half=half: half)
        got.append(ops.gemm_stream(x, w, offsets=off, a_rows=rows, scale=scale, rows=m + 3)[:m])
    assert torch.equal(*got)


@pytest.mark.parametrize("dt", DT)
def test_squared_relu_keeps_what_is_not_a_number(ops, dt):
    """Of plain numbers, infinities and NaN what torch gives, as a launch of its own and behind the product of a few rows."""
    x = torch.cat([_rand(300, dt=dt, seed=1), torch.tensor([0.0, -0.0, math.inf, -math.inf, math.nan, -math.nan], dtype=dt, device=DEV)])
    got, want = ops.relu2(x), (torch.relu(x.float()) ** 2).to(dt)
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.nan_to_num(7.0), want.nan_to_num(7.0))
    rows, w = _rand(7, 256, dt=torch.bfloat16, seed=2), _rand(2, 64, 256, dt=torch.bfloat16, seed=3)
    rows[4, 100] = math.nan
    off = torch.tensor([0, 3, 7], dtype=torch.int32, device=DEV)
    got = ops.gemm_few(rows, w, offsets=off, relu2=True)
    assert bool(got[4].isnan().all())
    assert torch.equal(got.isnan().any(1), torch.arange(7, device=DEV) == 4) and bool((got[5] > 0).any())


@pytest.mark.parametrize("way", ["passes", "cut", "wide", "half"])
def test_squared_relu_behind_the_weight_streaming_product(ops, monkeypatch, way):
    """The bits of the product and the activation as launches of their own, by every kernel that takes such rows."""
    from jax_llm_examples_amd.ops.layout import tile_
    counts, nout, k = [3, 0, 200, 70], 272, 4096
    x, w = _rand(sum(counts), k, dt=torch.bfloat16, seed=1), _rand(4, nout, k, dt=torch.bfloat16, scale=0.02, seed=2)
    x[5, 7], x[9] = float("nan"), 0.0
    tile_(w)
    off = torch.tensor([0] + counts).cumsum(0).int().to(DEV)
    monkeypatch.setattr(ops, "stream_wide", lambda *a: way == "wide")
    monkeypatch.setattr(ops, "stream_half", lambda *a: way == "half")
    monkeypatch.setattr(ops, "stream_cuts", lambda *a: (2, 3) if way == "cut" else (0, 1))
    got = ops.gemm_stream(x, w, offsets=off, relu2=True)
    want = ops.relu2(ops.gemm_stream(x, w, offsets=off))
    assert torch.equal(got.view(torch.int16), want.view(torch.int16)) and bool(got[5].isnan().all()) and not got[9].any()
    others = torch.cat([got[:5], got[10:]])
    assert not others.isnan().any() and bool((others > 0).any()) and bool((others == 0).any())


@pytest.mark.parametrize("counts,nout,k,cut,cuts", [
    ([77], 2048, 16384, 8, 8),                       # one group, all of it is cut
    ([192], 272, 4352, 2, 4),                        # pieces of unequal length, a second block of W of one tile
    ([33], 4096, 4096, 1, 3),                        # the last block alone
    ([5, 0, 192, 193, 31, 385], 800, 2048, 1, 2),    # groups without rows, with one, two and three passes; fifteen tiles and three
    ([5, 0, 192, 193, 31, 385], 800, 2048, 4, 7),    # all blocks
    ([1, 47, 17] * 50, 528, 1024, 2, 4),             # more groups than a look takes; pieces of a round of stages
    ([0, 0], 272, 1024, 1, 2)])                      # no rows at all
def test_blocks_cut_along_k_of_the_weight_streaming_product(ops, monkeypatch, counts, nout, k, cut, cuts):
    """One group with and without offsets, picked and scaled rows, float32 and bfloat16 results."""
    from jax_llm_examples_amd.ops.layout import tile_
    m, e = sum(counts), len(counts)
    x, w = _rand(m + 3, k, dt=torch.bfloat16, seed=1), _rand(e, nout, k, dt=torch.bfloat16, scale=0.02, seed=2)
    stored = w.clone()
    tile_(stored)
    off = torch.tensor([0] + counts).cumsum(0).int().to(DEV)
    rows = torch.randperm(m + 3, generator=torch.Generator().manual_seed(3))[:m].int().to(DEV)
    scale = _rand(m, seed=4)
    monkeypatch.setattr(ops, "stream_wide", lambda *a: False)
    monkeypatch.setattr(ops, "stream_half", lambda *a: False)
    monkeypatch.setattr(ops, "stream_cuts", lambda *a: (cut, cuts))
    m = max(m, 7)  # (rows that no group has are left as they are)
    args = dict(offsets=off, a_rows=rows, scale=scale, rows=m)
    got, low = (ops.gemm_stream(x, stored, out_f32=f, **args) for f in (True, False))
    assert torch.equal(got, ops.gemm_stream(x, stored, out_f32=True, **args)) or m > sum(counts)
    assert torch.equal(low[: sum(counts)], got[: sum(counts)].bfloat16())
    if e == 1:
        assert torch.equal(got, ops.gemm_stream(x[rows.long()], stored[0], out_f32=True) * scale[:, None])
    monkeypatch.setattr(ops, "stream_cuts", lambda *a: (0, 1))
    uncut = ops.gemm_stream(x, stored, out_f32=True, **args)
    o, from_cut = 0, (-(-nout // 256) - cut) * 256
    assert torch.equal(got[: sum(counts), :from_cut], uncut[: sum(counts), :from_cut])
    for c, we in zip(counts, w):
        want = x[rows[o: o + c].long()].double() @ we.double().T.contiguous() * scale[o: o + c, None].double()
        # float32 sums of k products of bfloat16 numbers: sqrt(k) 2^-24 of the terms' size is 8e-6 at 16,384 in the worst
        # order and a tenth of that as the matrix units add up
        for y in (got, uncut) if c else ():
            assert float((y[o: o + c].double() - want).norm() / want.norm()) <= 4e-6
        o += c


@pytest.mark.parametrize("swiglu", [False, True])
@pytest.mark.parametrize("counts", [[3] * 257, [3, 0, 200] * 50, [100] * 8, [3] + [120] * 20, [190] * 8, [3] + [400] * 40])
def test_experts_products_of_a_row_do_not_depend_on_how_the_others_are_shared_out(ops, counts, swiglu):
    """The first expert's rows beside full groups, beside empty ones and one that has all the rows, beside odd ones: the same bits."""
    from jax_llm_examples_amd.ops.layout import tile_
    nout, k, first, rest = 544, 4096, counts[0], sum(counts[1:])
    x = _rand(sum(counts), k, dt=torch.bfloat16, seed=1)
    w = _rand(1, nout, k, dt=torch.bfloat16, scale=0.02, seed=2).repeat(len(counts), 1, 1)
    tile_(w)
    got = []
    for others in (counts[1:], [0] * (len(counts) - 2) + [rest], [rest // 3] + [0] * (len(counts) - 3) + [rest - rest // 3]):
        off = torch.tensor([0, first] + others).cumsum(0).int().to(DEV)
        got.append(ops.gemm_stream(x, w, offsets=off, swiglu=swiglu)[:first])
    assert torch.equal(got[0], got[1]) and torch.equal(got[0], got[2])


@pytest.mark.parametrize("counts,nout,k,swiglu", [
    ([5, 0, 192, 193, 31, 385], 272, 4096, False),   # several passes, two blocks of W, the second of one tile
    ([200, 190, 260, 385, 193], 272, 512, False),    # passes that differ from the first group's two by one: pass after pass
    ([410, 577, 500], 2336, 256, True),              # the same with three and four, the last group's blocks in the last round
    ([190, 385, 260, 385, 193], 2048, 256, False),   # the same with blocks of W for every die
    ([100, 33, 64], 544, 4352, True),                # one pass a group
    ([3] * 257, 64, 4096, False),                    # more groups than compute units
    ([200] * 65, 512, 1024, True)])                  # more groups than a look takes, two passes each
def test_passes_of_the_weight_streaming_product_against_64_bits(ops, monkeypatch, counts, nout, k, swiglu):
    from jax_llm_examples_amd.ops.layout import tile_
    m, e = sum(counts), len(counts)
    x, w = _rand(m + 3, k, dt=torch.bfloat16, seed=1), _rand(e, nout, k, dt=torch.bfloat16, scale=0.02, seed=2)
    stored = w.clone()
    tile_(stored)
    off = torch.tensor([0] + counts).cumsum(0).int().to(DEV)
    rows = torch.randperm(m + 3, generator=torch.Generator().manual_seed(3))[:m].int().to(DEV)
    scale = _rand(m, seed=4)
    monkeypatch.setattr(ops, "stream_wide", lambda *a: False)
    monkeypatch.setattr(ops, "stream_half", lambda *a: False)
    got = ops.gemm_stream(x, stored, offsets=off, a_rows=rows, scale=scale, swiglu=swiglu, rows=m, out_f32=True)
    o = 0
    for c, we in zip(counts, w):
        want = x[rows[o: o + c].long()].double() @ we.double().T.contiguous() * scale[o: o + c, None].double()
        if swiglu:
            want = torch.nn.functional.silu(want[:, : nout // 2]) * want[:, nout // 2:]
        if c:  # (see above; the activation doubles it)
            assert float((got[o: o + c].double() - want).norm() / want.norm()) <= 4e-6
        o += c


def test_rows_off_their_16_bytes_take_the_passes(ops, monkeypatch):
    """Rows that begin at 8 bytes, where the wide tiles want 16."""
    from jax_llm_examples_amd.ops.layout import tile_
    x, w = _rand(400, 256, dt=torch.bfloat16, seed=1), _rand(1, 64, 256, dt=torch.bfloat16, scale=0.1, seed=2)
    tile_(w)
    off = torch.tensor([0, 400], dtype=torch.int32, device=DEV)
    elsewhere = torch.empty(400 * 256 + 4, dtype=torch.bfloat16, device=DEV)[4:].view(400, 256)
    elsewhere.copy_(x)
    monkeypatch.setattr(ops, "stream_wide", lambda *a: True)
    got = [ops.gemm_stream(t, w, offsets=off) for t in (x, elsewhere)]
    assert torch.equal(*got)


@pytest.mark.parametrize("dt", DT)
@pytest.mark.parametrize("d", [48, 50, 320, 1024, 2048, 4104, 8192])
def test_shift_apart_from_its_norm(ops, dt, d):
    """With many rows the shift is a kernel of its own behind the sums: the bits of the kernel that does both, at segments
    that begin and end within, at and across its blocks, with and without a branch output."""
    import types
    from jax_llm_examples_amd.parts.residual import GatedBranch
    lens, starts = [1, 7, 8, 30, 3, 17], [5, 0, 3, 0, 0, 9]
    n, cu = sum(lens), torch.tensor([0] + lens).cumsum(0)
    i32 = lambda v: torch.as_tensor(v, dtype=torch.int32).to(DEV)
    ctx = types.SimpleNamespace(positions=i32([s + t for s, k in zip(starts, lens) for t in range(k)]),
                                token_segment=i32([i for i, k in enumerate(lens) for _ in range(k)]), cu_seqlens=i32(cu),
                                state_slots=i32([3, 0, 5, 1, 2, 4]), state_phase=i32([0, 1, 1, 0, 0, 1]))
    x, y, g = _rand(n, d, seed=1), _rand(n, d, dt=dt, seed=2), _rand(n, d, dt=dt, seed=3)
    v = [_rand(d, seed=4 + i) for i in range(5)]
    for delta in (None, y, GatedBranch(y, v[0], g, v[1], v[2], 1e-3)):
        got = []
        for apart in (1 << 62, 1):
            ops.SHIFT_APART = (apart,) * 3
            state = _rand(6, 2, d, seed=9)
            got.append((*ops.add_norm_shift(x.clone(), delta, v[3], 1e-5, dt, (v[4], state), ctx), state))
        del ops.SHIFT_APART
        for a, b, what in zip(*got, ("sums", "normed rows", "shifted rows", "state")):
            assert torch.equal(a, b), (what, float((a - b).abs().max()))


@pytest.mark.parametrize("dt", DT)
@pytest.mark.parametrize("off", [0, 1])
@pytest.mark.parametrize("d", [63, 100, 126, 510, 512, 1000, 1026, 1032, 2050, 4092, 4098, 4100, 8188, 8190])
def test_gated_branch_norm_and_shift_at_odd_widths(ops, dt, d, off):
    """Every form of the sandwich arrangement's kernel against its definition in 64 bits: rows in pieces of four and of one,
    one or several a thread, weights that lie at any float; with the shift in the same kernel and apart."""
    import types
    from jax_llm_examples_amd.parts.residual import GatedBranch
    lens, starts = [1, 7, 12], [5, 0, 3]
    n, cu = sum(lens), torch.tensor([0] + lens).cumsum(0)
    i32 = lambda v: torch.as_tensor(v, dtype=torch.int32).to(DEV)
    ctx = types.SimpleNamespace(positions=i32([s + t for s, k in zip(starts, lens) for t in range(k)]),
                                token_segment=i32([i for i, k in enumerate(lens) for _ in range(k)]), cu_seqlens=i32(cu),
                                state_slots=i32([2, 0, 1]), state_phase=i32([0, 1, 1]))
    x, y, g = _rand(n, d, seed=1), _rand(n, d, dt=dt, seed=2), _rand(n, d, dt=dt, seed=3)
    v = [_rand(d + off, seed=4 + i)[off:] for i in range(5)]
    y64 = (y.double() + v[0].double()) * torch.sigmoid(g.double() + v[1].double())
    sums = x.double() + y64 / torch.sqrt((y64 * y64).mean(-1, keepdim=True) + 1e-3) * v[2].double()
    h = sums / torch.sqrt((sums * sums).mean(-1, keepdim=True) + 1e-5) * v[3].double()
    old = _rand(3, 2, d, seed=9).double()
    before = torch.cat([old[2, 0][None], torch.zeros(1, d, dtype=torch.float64, device=DEV), h[1:7], old[1, 1][None], h[8:19]])
    new = old.clone()
    new[2, 1], new[0, 0], new[1, 0] = h[0], h[7], h[19]
    for apart in (1 << 62, 1):
        ops.SHIFT_APART = (apart,) * 3
        state = _rand(3, 2, d, seed=9)
        got = (*ops.add_norm_shift(x.clone(), GatedBranch(y, v[0], g, v[1], v[2], 1e-3), v[3], 1e-5, dt, (v[4], state), ctx), state)
        del ops.SHIFT_APART
        for a, b, what in zip(got, (sums, h, h + (before - h) * v[4].double(), new), ("sums", "rows", "shifted", "state")):
            # float32 arithmetic, some ten roundings and two sums; rows rounded to the run dtype
            tol = 2e-6 if a.dtype == torch.float32 else 2.0 ** -8
            assert float((a.double() - b).norm() / b.norm()) < tol, (what, apart)


@pytest.mark.parametrize("dt", DT)
@pytest.mark.parametrize("off", [0, 1])
@pytest.mark.parametrize("f", [100, 4092, 4100, 8192, 14340, 16384, 16388, 1001])
def test_polynomial_activation_at_odd_widths(ops, dt, f, off):
    """Every form of the kernel (pieces of eight, four and one, the row kept or read twice), the bias at any float."""
    z, b, c = _rand(5, f, dt=dt, seed=1), _rand(f + off, seed=2)[off:], _rand(4, seed=3)
    u = z.double() + b.double()
    norm = lambda t: t / torch.sqrt((t * t).mean(-1, keepdim=True) + 1e-4)
    c64 = c.double()
    want = c64[0] * norm(u) + c64[1] * norm(u ** 2) + c64[2] * norm(u ** 3) + c64[3]
    got = ops.polynorm(z, b, c, 1e-4)
    assert float((got.double() - want).norm() / want.norm()) < (2e-6 if dt == torch.float32 else 2.0 ** -8)


@pytest.mark.parametrize("n,d,f,e,k", [(300, 128, 48, 16, 1), (700, 264, 72, 3, 2), (2048, 512, 256, 16, 1),
                                       (150, 64, 40, 128, 1)])
def test_grouped_product_for_many_rows(ops, ref, n, d, f, e, k):
    dt = torch.bfloat16
    h = _rand(n, d, dt=dt, seed=1)
    wgu = _rand(e, 2 * f, d, dt=dt, scale=0.1, seed=2)
    wd = _rand(e, d, f, dt=dt, scale=0.1, seed=3)
    g = torch.Generator().manual_seed(5)
    ids = torch.stack([torch.randperm(e, generator=g)[:k] for _ in range(n)]).to(torch.int32).to(DEV)
    if n == 300:
        ids[:200] = 3  # one expert with more rows than one block, others with none
    gates = torch.rand(n, k, generator=g).to(DEV)
    off, tok, gate, inv = ops.moe_align(ids, gates, e)
    act = ops.gemm_grouped(h, wgu, offsets=off, a_rows=tok, scale=gate, swiglu=True)
    gu = ops.gemm(h, wgu, offsets=off, a_rows=tok, scale=gate, out_f32=True)  # the general kernel, float32 result
    want = torch.nn.functional.silu(gu[:, :f]) * gu[:, f:]
    assert act.shape == (n * k, f)
    assert float((act.float() - want).abs().max() / want.abs().max()) <= 5e-3
    plain = ops.gemm_grouped(h, wgu, offsets=off, a_rows=tok, scale=gate, out_f32=True)
    assert float((plain - gu).abs().max() / gu.abs().max()) <= 2e-5
    down = ops.gemm_grouped(act, wd, offsets=off)
    want_d = ops.gemm(act, wd, offsets=off, out_f32=True)
    assert float((down.float() - want_d).abs().max() / want_d.abs().max()) <= 5e-3
    # the whole expert layer at this size takes the same path
    _assert_close_to_scale(ops.materialize(ops.moe_experts(h, ids, gates, wgu, wd, None)),
                           ref.moe_experts(h, ids, gates, wgu, wd, None), dt)
    dense = ops.gemm_grouped(h, wgu[0], out_f32=True)  # one group, no offsets
    assert float((dense - h.float() @ wgu[0].float().t()).abs().max() / dense.abs().max()) <= 2e-5
    head = ops.lm_head(h[:100, :], _rand(311, d, dt=dt, seed=7))
    assert head.dtype == torch.float32 and head.shape == (100, 311)


@pytest.mark.parametrize("n,d,f,e,k", [(300, 256, 32, 16, 1), (700, 768, 96, 3, 2), (2048, 512, 256, 16, 1),
                                       (150, 256, 48, 128, 1), (900, 256, 80, 2, 1)])
def test_weight_streaming_grouped_product(ops, ref, n, d, f, e, k):
    """Groups without rows, with a few, with more than one pass of 192; an odd number of weight tiles."""
    from jax_llm_examples_amd.ops.layout import tile_
    dt = torch.bfloat16
    h = _rand(n, d, dt=dt, seed=1)
    wgu = _rand(e, 2 * f, d, dt=dt, scale=0.1, seed=2)
    wd = _rand(e, d, f, dt=dt, scale=0.1, seed=3)
    g = torch.Generator().manual_seed(5)
    ids = torch.stack([torch.randperm(e, generator=g)[:k] for _ in range(n)]).to(torch.int32).to(DEV)
    if n == 300:
        ids[:270] = 3  # one expert with more rows than one pass, others with none
    gates = torch.rand(n, k, generator=g).to(DEV)
    off, tok, gate, inv = ops.moe_align(ids, gates, e)
    wgu_t = wgu.clone()
    tile_(wgu_t)
    gu = ops.gemm(h, wgu, offsets=off, a_rows=tok, scale=gate, out_f32=True)  # the general kernel, float32 result
    plain = ops.gemm_stream(h, wgu_t, offsets=off, a_rows=tok, scale=gate, out_f32=True)
    assert float((plain - gu).abs().max() / gu.abs().max()) <= 2e-5
    if f % 16 == 0:
        act = ops.gemm_stream(h, wgu_t, offsets=off, a_rows=tok, scale=gate, swiglu=True)
        want = torch.nn.functional.silu(gu[:, :f]) * gu[:, f:]
        assert act.shape == (n * k, f)
        assert float((act.float() - want).abs().max() / want.abs().max()) <= 5e-3
    else:
        with pytest.raises(Exception, match="refuses|needs"):
            ops.gemm_stream(h, wgu_t, offsets=off, a_rows=tok, scale=gate, swiglu=True)
        act = ops.gemm_grouped(h, wgu, offsets=off, a_rows=tok, scale=gate, swiglu=True)
    if f % 256 == 0:
        wd_t = wd.clone()
        tile_(wd_t)
        down = ops.gemm_stream(act, wd_t, offsets=off)
        want_d = ops.gemm(act, wd, offsets=off, out_f32=True)
        assert float((down.float() - want_d).abs().max() / want_d.abs().max()) <= 5e-3
    dense = ops.gemm_stream(h, wgu_t[0], out_f32=True)  # one group, no offsets
    assert float((dense - h.float() @ wgu[0].float().t()).abs().max() / dense.abs().max()) <= 2e-5
    with pytest.raises(Exception, match="refuses|needs"):
        ops.gemm_stream(h[:, :d - 128].contiguous(), wgu_t[:, :, :d - 128].contiguous())


def test_streaming_layout_gives_the_same_results_bit_for_bit(ops):
    from jax_llm_examples_amd.ops.layout import can_tile, tile_, untiled
    dt = torch.bfloat16
    w = _rand(3, 96, 160, dt=dt, seed=1)
    wt = w.clone()
    assert can_tile(w) and not can_tile(_rand(3, 90, 160, dt=dt)) and not can_tile(w.float())
    tile_(wt)
    assert not torch.equal(wt, w) and torch.equal(untiled(wt), w)
    first_tile = wt[1].flatten()[:512].reshape(4, 16, 8)  # the first kilobyte: rows 0..15, k 0..31 as [g][r][8]
    assert torch.equal(first_tile[2, 5], w[1, 5, 16:24])
    second = wt[1].flatten()[512:1024].reshape(4, 16, 8)  # the next tile goes on along K
    assert torch.equal(second[0, 3], w[1, 3, 32:40])
    for n, d, f, e, k in [(8, 128, 48, 16, 1), (50, 160, 96, 5, 2), (400, 256, 64, 4, 1)]:
        h = _rand(n, d, dt=dt, seed=1)
        wgu, wd = _rand(e, 2 * f, d, dt=dt, scale=0.1, seed=2), _rand(e, d, f * 1, dt=dt, scale=0.1, seed=3)
        if f % 32:
            continue
        g = torch.Generator().manual_seed(5)
        ids = torch.stack([torch.randperm(e, generator=g)[:k] for _ in range(n)]).to(torch.int32).to(DEV)
        gates = torch.rand(n, k, generator=g).to(DEV)
        wgu_t, wd_t = wgu.clone(), wd.clone()
        tile_(wgu_t), tile_(wd_t)
        a = ops.materialize(ops.moe_experts(h, ids, gates, wgu, wd, None))
        b = ops.materialize(ops.moe_experts(h, ids, gates, wgu_t, wd_t, None, tiled=True))
        assert torch.equal(a, b)
    for m in (3, 40, 200):
        h, w2 = _rand(m, 160, dt=dt, seed=4), _rand(17 * 16, 160, dt=dt, seed=5)  # an odd number of row tiles
        w2t = w2.clone()
        tile_(w2t)
        assert torch.equal(ops.lm_head(h, w2), ops.lm_head(h, w2t, tiled=True))


@pytest.mark.parametrize("m,v", [(1, 1), (3, 512), (2, 8191), (5, 8192), (64, 8200), (2, 32767), (3, 32768), (2, 32772), (2, 32773), (1, 202048)])
@pytest.mark.parametrize("off", [0, 1])
def test_greedy_rows_and_their_copy(ops, m, v, off):
    """Edges of what a block takes of a long row (8,192) and of the longest row that one block takes alone (32,768), rows that do not start at 16
    bytes; equal maxima, rows without any number and rows of the lowest value."""
    g = torch.Generator().manual_seed(v)
    flat = torch.empty(m * v + off, device=DEV)
    logits = flat[off:].view(m, v)
    logits.copy_(torch.randn(m, v, generator=g))
    logits[0, v // 3] = logits[0, v - 1] = 9.0
    if m > 1:
        logits[1] = float("-inf")
    if m > 2:
        logits[2] = float("nan")
        logits[2, v // 2] = -7.0
    want = [v // 3] + [0] * (m > 1) + [v // 2] * (m > 2) + torch.argmax(logits[3:].cpu(), -1).tolist()
    got, kept = ops.greedy(logits, copy=True)
    assert got == want and torch.equal(kept.view(torch.int32), logits.contiguous().view(torch.int32))
    assert ops.greedy(logits) == (want, None)


@pytest.mark.parametrize("n,d", [(1, 64), (3, 2048), (2, 2056), (5, 100), (70, 5120)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_embedding_rows_times_a_number(ops, ref, n, d, dtype):
    table = torch.randn(90, d, generator=torch.Generator().manual_seed(d)).to(DEV, dtype)
    tok = torch.randint(0, 90, (n,), generator=torch.Generator().manual_seed(n)).int().to(DEV)
    for mul in (1.0, 45.254834):
        assert torch.equal(ops.embed(tok, table, mul), ref.embed(tok, table, mul))


@pytest.mark.parametrize("n,d", [(1, 8), (257, 8), (300, 264), (31, 2048), (513, 2056)])
def test_embedding_rows_end_within_a_block(ops, ref, n, d):
    table = torch.randn(600, d, generator=torch.Generator().manual_seed(d)).to(DEV, torch.bfloat16)
    tok = torch.randint(0, 600, (n,), generator=torch.Generator().manual_seed(n)).int().to(DEV)
    assert torch.equal(ops.embed(tok, table, 1.5), ref.embed(tok, table, 1.5))


@pytest.mark.parametrize("k,shared,own", [(1, True, False), (2, False, False), (2, True, True), (6, True, False)])
def test_chosen_rows_of_an_expert_sum_stay_in_pieces(ops, k, shared, own):
    from jax_llm_examples_amd.ops.hip import ExpertSum

    g = torch.Generator().manual_seed(k)
    n, d = 9, 2048
    bf = lambda *s: torch.randn(*s, generator=g).to(DEV, torch.bfloat16)
    inv = torch.randperm(n * k, generator=g).int()
    if own:
        inv[::3] = -1
    lazy = ExpertSum(bf(n * k, d), inv.to(DEV), k, bf(n, d) if shared else None, n, d,
                     (bf(n, d), torch.rand(n, k, generator=g).to(DEV)) if own else None)
    idx = torch.tensor([7, 0, 7, 3], dtype=torch.int32, device=DEV)
    x = torch.randn(n, d, generator=g).to(DEV)
    w = torch.rand(d, generator=g).to(DEV)
    a, b = ops.gather_rows(x, idx), x.clone()
    got, _ = ops.add_rmsnorm(a, lazy.rows(ops, idx), w, 1e-5, torch.bfloat16)
    want, _ = ops.add_rmsnorm(b, lazy, w, 1e-5, torch.bfloat16)
    assert torch.equal(a, b[idx.long()]) and torch.equal(got, want[idx.long()])


def _few_bound(a, b):
    """What float32 sums of exact products may be off by, a k of any order: (k + 2) roundings of 2^-24 of the sum of their sizes."""
    return (a.shape[1] + 2) * 2.0 ** -24 * (a.double().abs() @ b.double().abs().t()) + 1e-30


@pytest.mark.parametrize("m,nout,k", [(1, 64, 64), (8, 70, 192), (16, 33, 128), (17, 96, 320), (33, 500, 256), (64, 130, 5120),
                                       (5, 1000, 8192), (3, 80, 1088), (64, 8192, 128), (24, 4112, 64), (63, 16, 448)])
@pytest.mark.parametrize("tiles", [0, 11, 12, 14, 21, 22, 24, 41, 42, 44])
def test_product_of_a_few_rows(ops, m, nout, k, tiles):
    """Tiles with one row and one column over, lines fewer than wavefronts, every tile of the choice."""
    from jax_llm_examples_amd.ops.layout import can_tile, tile_

    g = torch.Generator().manual_seed(m + nout)
    a = torch.randn(m, k, generator=g).to(DEV, torch.bfloat16)
    b = torch.randn(nout, k, generator=g).to(DEV, torch.bfloat16)
    want = a.double() @ b.double().t()
    got = ops.gemm_few(a, b, out_f32=True, tiles=tiles)
    assert ((got.double() - want).abs() <= _few_bound(a, b)).all()
    assert torch.equal(ops.gemm_few(a, b, tiles=tiles), got.bfloat16())
    # (a row's sums are formed in one order whatever the tiles, the other rows and the layout)
    assert torch.equal(ops.gemm_few(a[m - 1:].contiguous(), b, out_f32=True)[0], got[m - 1])
    if can_tile(b):
        bt = b.clone()
        tile_(bt)
        assert torch.equal(ops.gemm_few(a, bt, out_f32=True, tiled=True, tiles=tiles), got)


@pytest.mark.parametrize("sizes", [[0, 17, 1, 0, 16], [33, 0, 64, 2, 30], [1, 0, 0, 0, 0], [0, 0, 0, 0, 3], [2] * 70 + [0] * 5 + [9]])
@pytest.mark.parametrize("tiled", [False, True])
def test_product_of_a_few_rows_in_groups(ops, sizes, tiled):
    """Groups without rows, group slots, the last group's matrix elsewhere and in the other layout, picked rows, a scale a row,
    and both activations."""
    from jax_llm_examples_amd.ops.layout import tile_

    g = torch.Generator().manual_seed(len(sizes))
    G, m, n, k, f = len(sizes), sum(sizes), 30, 256, 96
    bf = lambda *s: torch.randn(*s, generator=g).to(DEV, torch.bfloat16)
    w, last, x = bf(G - 1, 2 * f, k), bf(2 * f, k), bf(n, k)
    off = torch.tensor([0] + sizes).cumsum(0).int().to(DEV)
    rows = torch.randint(0, n, (m,), generator=g).int().to(DEV)
    scale = torch.rand(m, generator=g).to(DEV)
    group = torch.repeat_interleave(torch.arange(G), torch.tensor(sizes)).to(DEV)
    every = torch.cat([w, last[None]]).double()
    xs = x[rows.long()].double()
    want = torch.einsum("mk,mnk->mn", xs, every[group]) * scale.double()[:, None]
    bound = (k + 3) * 2.0 ** -24 * torch.einsum("mk,mnk->mn", xs.abs(), every[group].abs()) * scale.double()[:, None] + 1e-30
    wt = w.clone()
    if tiled:
        tile_(wt)
    kw = dict(offsets=off, a_rows=rows, scale=scale, tiled=tiled, b_last=last)
    got = ops.gemm_few(x, wt, out_f32=True, **kw)
    assert ((got.double() - want).abs() <= bound).all()
    # (a factor of 2^-8 for the rounding to bfloat16, before and after the square)
    y = ops.gemm_few(x, wt, relu2=True, **kw)
    assert torch.equal(y, (got.bfloat16().float().clamp(min=0) ** 2).bfloat16())
    for act in (1, 2):
        y = ops.gemm_few(x, wt, swiglu=act, out_f32=True, **kw)
        gate, up, of_gate, of_up = want[:, :f], want[:, f:], bound[:, :f], bound[:, f:]
        ref_act = torch.nn.functional.silu(gate) if act == 1 else torch.nn.functional.gelu(gate, approximate="tanh")
        # (the sums' own bounds, through slopes of up to 1.13; expf and tanhf within a few units of 2^-24 of 1 + |x|)
        tol = 1.13 * of_gate * (up.abs() + of_up) + ref_act.abs() * of_up + 32 * 2.0 ** -24 * (1 + gate.abs()) * up.abs()
        assert ((y.double() - ref_act * up).abs() <= tol + 1e-30).all()


@pytest.mark.parametrize("tiles", [12, 14, 22, 24, 42, 44])
@pytest.mark.parametrize("sizes", [None, [0, 17, 64, 1, 33]])
@pytest.mark.parametrize("f,tiled", [(48, False), (48, True), (80, True), (88, False)])
def test_gate_and_up_of_a_few_rows_with_every_tile(ops, f, tiled, sizes, tiles):
    """The last block part of its tiles of gate rows and of up rows, whole tiles and half of one; one matrix, or groups of
    which one fills the largest tile of rows."""
    from jax_llm_examples_amd.ops.layout import tile_

    g = torch.Generator().manual_seed(f)
    G, m, k = len(sizes or [1]), sum(sizes or [50]), 192
    w, x = (torch.randn(*s, generator=g).to(DEV, torch.bfloat16) for s in ((G, 2 * f, k), (m, k)))
    group = torch.repeat_interleave(torch.arange(G), torch.tensor(sizes or [m])).to(DEV)
    want = torch.stack([x[t].double() @ w[group[t]].double().t() for t in range(m)])
    bound = torch.stack([(k + 3) * 2.0 ** -24 * (x[t].double().abs() @ w[group[t]].double().abs().t()) for t in range(m)])
    wt = w.clone()
    if tiled:
        tile_(wt)
    kw = dict(tiled=tiled, tiles=tiles, offsets=None if sizes is None else torch.tensor([0] + sizes).cumsum(0).int().to(DEV))
    for act in (1, 2):
        y = ops.gemm_few(x, wt if sizes else wt[0], swiglu=act, out_f32=True, **kw)
        gate, up, of_gate, of_up = want[:, :f], want[:, f:], bound[:, :f], bound[:, f:]
        ref_act = torch.nn.functional.silu(gate) if act == 1 else torch.nn.functional.gelu(gate, approximate="tanh")
        # (the sums' own bounds, through slopes of up to 1.13; expf and tanhf within a few units of 2^-24 of 1 + |x|)
        tol = 1.13 * of_gate * (up.abs() + of_up) + ref_act.abs() * of_up + 32 * 2.0 ** -24 * (1 + gate.abs()) * up.abs()
        assert ((y.double() - ref_act * up).abs() <= tol + 1e-30).all()


@pytest.mark.parametrize("tiles", [11, 12, 14, 21, 22, 24, 41, 42, 44])
@pytest.mark.parametrize("nout,tiled", [(80, True), (70, False)])
def test_grouped_product_of_a_few_rows_with_every_tile(ops, nout, tiled, tiles):
    from jax_llm_examples_amd.ops.layout import tile_

    g = torch.Generator().manual_seed(nout)
    sizes, k = [0, 17, 64, 1, 33, 65], 320
    m = sum(sizes)
    w, x = (torch.randn(*s, generator=g).to(DEV, torch.bfloat16) for s in ((len(sizes), nout, k), (m, k)))
    off = torch.tensor([0] + sizes).cumsum(0).int().to(DEV)
    wt = w.clone()
    if tiled:
        tile_(wt)
    got = ops.gemm_few(x, wt, offsets=off, tiled=tiled, tiles=tiles, out_f32=True)
    for e, (lo, hi) in enumerate(zip(off[:-1].tolist(), off[1:].tolist())):
        want = x[lo:hi].double() @ w[e].double().t()
        assert ((got[lo:hi].double() - want).abs() <= _few_bound(x[lo:hi], w[e])).all()


@pytest.mark.parametrize("m,nout,k,groups,swiglu,grouped,tiled,tiles", [
    (2, 5120, 8192, 17, 0, 1, 1, 11), (6, 2048, 4096, 9, 0, 1, 1, 11), (30, 5120, 8192, 17, 0, 1, 1, 11),  # a few rows a group
    (16, 4096, 1408, 64, 0, 1, 1, 12), (128, 7168, 2048, 16, 0, 1, 1, 12), (128, 4096, 2048, 8, 0, 1, 1, 22),
    (95, 14336, 4096, 8, 1, 1, 1, 12), (96, 14336, 4096, 8, 1, 1, 1, 22), (106, 14336, 4096, 4, 1, 1, 1, 22), (108, 14336, 4096, 4, 1, 1, 1, 44),
    (2, 16384, 5120, 17, 1, 1, 1, 12), (1, 16384, 5120, 1, 1, 0, 0, 14),
    (1, 50000, 3072, 1, 0, 0, 1, 12), (8, 16000, 2048, 1, 0, 0, 1, 12), (1, 202048, 5120, 1, 0, 0, 0, 12),  # many rounds
    (1, 32000, 2048, 1, 0, 0, 0, 14), (1, 2048, 2048, 1, 0, 0, 0, 11), (64, 202048, 5120, 1, 0, 0, 1, 44)])
def test_tiles_of_a_product_of_a_few_rows(ops, m, nout, k, groups, swiglu, grouped, tiled, tiles):
    assert ops._query("jle_gemm_few_tiles", m, nout, k, groups, swiglu, grouped, tiled) == tiles


def test_product_of_a_few_rows_refuses_what_it_cannot_read(ops):
    from jax_llm_examples_amd.ops.hip import KernelError

    a, b = torch.zeros(4, 64, device=DEV, dtype=torch.bfloat16), torch.zeros(16, 64, device=DEV, dtype=torch.bfloat16)
    odd = torch.zeros(4 * 64 + 1, device=DEV, dtype=torch.bfloat16)[1:].view(4, 64)
    for x, w in ((a[:, :56].contiguous(), b[:, :56].contiguous()), (odd, b)):
        assert not ops._few(x, w)
        with pytest.raises(KernelError):
            ops.gemm_few(x, w)
    assert torch.equal(ops.linear(odd, b), torch.zeros(4, 16, device=DEV, dtype=torch.bfloat16))


@pytest.mark.parametrize("counts,nout,k", [
    ([1, 0, 63, 64, 65, 128, 129, 160], 96, 256),
    ([287, 288, 289, 576, 577, 256, 257, 700, 1], 144, 512),  # one, two and three tiles of rows, a second block of W of one tile
    ([3, 0, 300] * 50, 64, 256),                              # more groups than a look takes
    ([192] * 8, 1168, 768)])                                  # more than eight blocks of W
def test_narrower_tiles_of_the_weight_streaming_product(ops, monkeypatch, counts, nout, k):
    """The bits of the kernel that takes a group's rows in passes, rows gathered and scaled."""
    from jax_llm_examples_amd.ops.layout import tile_
    m, e = sum(counts), len(counts)
    x, w = _rand(m + 3, k, dt=torch.bfloat16, seed=1), _rand(e, nout, k, dt=torch.bfloat16, scale=0.1, seed=2)
    tile_(w)
    off = torch.tensor([0] + counts).cumsum(0).int().to(DEV)
    rows = torch.randperm(m + 3, generator=torch.Generator().manual_seed(3))[:m].int().to(DEV)
    scale = _rand(m, seed=4)
    got = []
    for half in (False, True):
        monkeypatch.setattr(ops, "stream_half", lambda *a, half=half: half, raising=False)
        monkeypatch.setattr(ops, "stream_wide", lambda *a: False, raising=False)
        got.append(ops.gemm_stream(x, w, offsets=off, a_rows=rows, scale=scale, rows=m))
    assert torch.equal(*got)


@pytest.mark.parametrize("d", [256, 260, 1024, 1028, 2048, 2052, 4096, 4100, 8192, 8196, 2050])
@pytest.mark.parametrize("k", [0, 1, 2, 3])
def test_sum_with_factors_by_pieces_of_four(ops, d, k):
    """Widths at the edges of the pieces a thread takes, and those that go element by element; a plain term (k = 0) or one to
    three pieces of an expert sum, a second term, a scale a channel."""
    from jax_llm_examples_amd.ops.hip import ExpertSum
    from jax_llm_examples_amd.parts.residual import ScaledSum

    g = torch.Generator().manual_seed(d + k)
    n = 5
    bf = lambda *s: torch.randn(*s, generator=g).to(DEV, torch.bfloat16)
    x, b = torch.randn(n, d, generator=g).to(DEV), bf(n, d)
    vec, w = (torch.rand(d, generator=g).to(DEV) + 0.5 for _ in range(2))
    if k:
        inv, rows = torch.randperm(n * k, generator=g).int().to(DEV), bf(n * k, d)
        a, plain = ExpertSum(rows, inv, k, None, n, d), rows.double()[inv.long()].view(n, k, d).sum(1)
    else:
        a = bf(n, d)
        plain = a.double()
    want = x.double() + vec.double() * (0.7 * plain + 1.3 * b.double())
    h, h32 = ops.scaled_add_norm(x, ScaledSum([(a, 0.7), (b, 1.3)], vec), w, 1e-5, torch.bfloat16, want32=True)
    normed = want / torch.sqrt((want ** 2).mean(-1, keepdim=True) + 1e-5) * w.double()
    # (a few roundings of 2^-24 of what is added up; the row's statistics another few)
    size = x.double().abs() + want.abs() + vec.double() * (0.7 * plain.abs() + 1.3 * b.double().abs()) + 4
    assert ((x.double() - want).abs() <= 8 * 2.0 ** -24 * size).all()
    assert ((h32.double() - normed).abs() <= 32 * 2.0 ** -24 * (size + normed.abs())).all()
    assert torch.equal(h, h32.bfloat16())


@pytest.mark.parametrize("d", [1024, 2048, 4096, 8192])
@pytest.mark.parametrize("k", [0, 2])
def test_sum_with_factors_of_rows_off_their_16_bytes(ops, d, k):
    """Widths of each number of pieces, a term that starts 8 bytes on: element by element, to the same bounds."""
    from jax_llm_examples_amd.ops.hip import ExpertSum
    from jax_llm_examples_amd.parts.residual import ScaledSum

    g = torch.Generator().manual_seed(d + k)
    n = 5
    off = lambda *s: torch.randn(math.prod(s) + 4, generator=g).to(DEV, torch.bfloat16)[4:].view(*s)
    x, b = torch.randn(n, d, generator=g).to(DEV), off(n, d)
    vec, w = (torch.rand(d, generator=g).to(DEV) + 0.5 for _ in range(2))
    if k:
        inv, rows = torch.randperm(n * k, generator=g).int().to(DEV), off(n * k, d)
        a, plain = ExpertSum(rows, inv, k, None, n, d), rows.double()[inv.long()].view(n, k, d).sum(1)
    else:
        a = off(n, d)
        plain = a.double()
    want = x.double() + vec.double() * (0.7 * plain + 1.3 * b.double())
    size = x.double().abs() + want.abs() + vec.double() * (0.7 * plain.abs() + 1.3 * b.double().abs()) + 4
    h, h32 = ops.scaled_add_norm(x, ScaledSum([(a, 0.7), (b, 1.3)], vec), w, 1e-5, torch.bfloat16, want32=True)
    normed = want / torch.sqrt((want ** 2).mean(-1, keepdim=True) + 1e-5) * w.double()
    # (a few roundings of 2^-24 of what is added up; the row's statistics another few)
    assert ((x.double() - want).abs() <= 8 * 2.0 ** -24 * size).all()
    assert ((h32.double() - normed).abs() <= 32 * 2.0 ** -24 * (size + normed.abs())).all()
    assert torch.equal(h, h32.bfloat16())


@pytest.mark.parametrize("tile", [(8, 8), (8, 7), (8, 6), (6, 8), (8, 5), (8, 4), (6, 4), (4, 5), (4, 4)])
def test_dense_product_of_many_rows(ops, tile):
    """Every tile: one row and eight columns over, one less, several tiles each way, one to six stages; with a bias."""
    bm, bn = 32 * tile[0], 32 * tile[1]
    for m, n, k in ((1, 8, 64), (bm, bn, 128), (bm + 1, bn + 8, 192), (2 * bm - 1, 2 * bn - 8, 256), (3 * bm + 17, 9 * bn + 16, 384)):
        g = torch.Generator().manual_seed(m + n + k)
        x = torch.randn(m, k, generator=g).to(DEV, torch.bfloat16)
        w = (torch.randn(n, k, generator=g) * k ** -0.5).to(DEV, torch.bfloat16)
        bias = torch.randn(n, generator=g).to(DEV, torch.bfloat16)
        want, sums = x.double() @ w.double().t(), (k + 2) * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t())
        for b in (None, bias):
            got = ops.gemm_dense(x, w, tile[0] * 16 + tile[1], b).double()
            y = want if b is None else want + b.double()
            assert ((got - y).abs() <= 2.0 ** -8 * y.abs() + sums + 2.0 ** -24 * y.abs() + 1e-30).all()
            again = ops.gemm_dense(x[m // 2:].contiguous(), w, 4 * 16 + 4, b)
            assert torch.equal(again.double(), got[m // 2:])  # (a row's sums have one order whatever the tile and the other rows)


def test_dense_product_keeps_what_is_not_a_number_in_its_row(ops):
    x, w = (torch.randn(300, 128, device=DEV).bfloat16() for _ in range(2))
    want = ops.gemm_dense(x, w[:296].contiguous(), 8 * 16 + 8)
    x[299, 5], x[7, 127] = math.nan, math.inf
    got = ops.gemm_dense(x, w[:296].contiguous(), 8 * 16 + 8)
    keep = torch.ones(300, dtype=torch.bool)
    keep[[7, 299]] = False
    assert got[299].isnan().all() and not got[7].isfinite().any() and torch.equal(got[keep], want[keep])


def _dense_calls(ops, monkeypatch):
    """The sizes that the kernel of many rows is called with from here on."""
    called, kernel = [], ops.gemm_dense
    monkeypatch.setattr(ops, "gemm_dense", lambda h, w, *a, **kw: (called.append((h.shape[0], *w.shape)), kernel(h, w, *a, **kw))[1])
    return called


def test_dense_products_replayed(ops, monkeypatch):
    """In a graph, pass after pass with other rows in between; the kernel of many rows is what the graph holds."""
    x, w = torch.randn(512, 1024, device=DEV).bfloat16(), torch.randn(2048, 1024, device=DEV).bfloat16()
    ops.linear(x, w)
    graph = torch.cuda.CUDAGraph()
    called = _dense_calls(ops, monkeypatch)
    with torch.cuda.graph(graph):
        y = ops.linear(x, w)
        z = ops.swiglu_linear(y[:, :1024].contiguous(), w)
    assert called == [(512, 2048, 1024)] * 2
    sums = lambda a: 2.0 ** -8 * (a.double() @ w.double().t()).abs() + 1026 * 2.0 ** -24 * (a.double().abs() @ w.double().abs().t())
    for _ in range(3):
        x.copy_(torch.randn(512, 1024, device=DEV))
        graph.replay()
        torch.cuda.synchronize()
        assert ((y.double() - x.double() @ w.double().t()).abs() <= sums(x)).all()
        assert torch.equal(y, ops.linear(x, w)) and torch.equal(z, ops.swiglu_linear(y[:, :1024].contiguous(), w))


def test_which_products_of_many_rows_are_the_dense_kernels(ops, monkeypatch):
    """Plain, with a bias, under the activation, and a latent's keys and values; not where a gradient is wanted or a mode looks on."""
    from torch.utils.flop_counter import FlopCounterMode
    from jax_llm_examples_amd.engine.batch import GroupContext
    called = _dense_calls(ops, monkeypatch)
    x, w = torch.randn(384, 512, device=DEV).bfloat16(), torch.randn(1024, 512, device=DEV).bfloat16()
    bias = torch.randn(1024, device=DEV).bfloat16()
    for call in (lambda: ops.linear(x, w), lambda: ops.linear_bias(x, w, bias)[0], lambda: ops.swiglu_linear(x, w)):
        del called[:]
        call()
        assert called == [(384, 1024, 512)]
    del called[:]
    ops.linear(x, w.requires_grad_())
    with torch.no_grad(), FlopCounterMode(display=False) as seen:
        ops.linear(x, w)
    assert not called and seen.get_total_flops() == 2 * 384 * 1024 * 512
    n, H, R, ps = 256, 4, 512, 16
    zeros = lambda *s: torch.zeros(*s, dtype=torch.bfloat16, device=DEV)
    table = torch.arange(n // ps, dtype=torch.int32, device=DEV).view(1, -1)
    pos, seg = torch.arange(n, dtype=torch.int32, device=DEV), torch.zeros(n, dtype=torch.int32, device=DEV)
    meta = GroupContext(block_table=None, slot_mapping=None, width=n // ps, retention=("all",), seg_lens=[n], seg_starts=[0])
    monkeypatch.setattr(ops, "LATENT_EXPAND_PAIRS", 0)
    assert ops.latent_attention_expanded(zeros(n, H, 192), 128, zeros(H * 128, R), zeros(H * 128, R), zeros(n // ps, ps, R),
                                         zeros(n // ps, ps, 64), table, pos, seg, None, 0.1, meta) is not None
    assert called == [(n, H * 128, R), (H * 128, n, R)]


@pytest.mark.parametrize("dt", DT)
@pytest.mark.parametrize("hq,hk,hv,dk,dv,page,ps", [(4, 2, 2, 128, 128, 128, 16), (2, 4, 2, 64, 136, 144, 16), (3, 3, 1, 96, 300, 320, 32), (2, 1, 1, 20, 12, 24, 8), (2, 4, 2, 256, 512, 512, 16)])
def test_heads_of_many_tokens_prepared(ops, dt, hq, hk, hv, dk, dv, page, ps):
    """Values written sixteen tokens at a time: what the same tokens give in calls of fewer than 256, in scattered slots of pages."""
    import types
    n = 259
    rows = _rand(n, (hq + hk) * dk + hv * dv, dt=dt, seed=1)
    rot = types.SimpleNamespace(inv_freq=_rand(dk // 4, seed=2).abs(), rotary_dim=dk // 4 * 2, magnitude=1.1, pairing="half")
    prep = types.SimpleNamespace(query_scale=None, norm_span="head", rotation=rot, norm_weight_q=_rand(dk, seed=3), norm_weight_k=None,
                                 norm_eps=1e-5, norm_first=True)
    slots = torch.randperm((n // ps + 3) * ps, generator=torch.Generator().manual_seed(4))[:n].int().to(DEV)
    positions = torch.arange(n, dtype=torch.int32, device=DEV)
    got = []
    for cuts in ((0, n), (0, 200, n)):
        pages = torch.full((n // ps + 3, 2, hk, ps, page), 7.0, dtype=dt, device=DEV)
        q = [ops.heads_prepare(rows[a:b], hq, hk, hv, dk, dv, page, prep, positions[a:b], pages, slots[a:b]) for a, b in zip(cuts, cuts[1:])]
        got.append((torch.cat(q), pages))
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])
    plain = torch.cat([ops.heads_prepare(rows[a:b], hq, hk, hv, dk, dv, page, prep, positions[a:b], None, None) for a, b in ((0, 3), (3, n))])
    assert torch.equal(plain, got[0][0])
    values = got[0][1][:, 1].reshape(-1, hk, page, ps)[(slots // ps).long(), :, :, (slots % ps).long()]  # [n, hk, page]
    want = rows[:, (hq + hk) * dk:].reshape(n, hv, dv).repeat_interleave(hk // hv, 1)
    assert torch.equal(values[..., :dv], want) and not values[..., dv:].any()


@pytest.mark.parametrize("n,dim,paged,rotary,bf16,bytes_", [
    (255, 64, 1, 1, 1, 512), (9, 128, 1, 1, 0, 512), (200, 256, 1, 1, 0, 1024), (255, 512, 1, 1, 1, 2048), (2048, 512, 0, 1, 0, 2048), (300, 128, 0, 0, 1, 0),
    (256, 128, 1, 1, 1, 4352), (256, 128, 1, 1, 0, 8704), (256, 512, 1, 1, 1, 8192), (256, 64, 1, 0, 1, 4352)])
def test_heads_take_the_shared_memory_of_what_a_block_does(ops, n, dim, paged, rotary, bf16, bytes_):
    """A wavefront of its own: its head and no room for others or for a value tile, so that 32 of them fit a compute unit's 160 KB."""
    assert ops._query("jle_heads_prepare_shared", n, dim, paged, rotary, bf16) == bytes_


def test_heads_of_more_tokens_than_a_launch_takes(ops):
    """2^26 heads and more: threads of two launches and a rest; the same as in calls of a part each."""
    import types
    n, hq, d, ps = (1 << 20) + 37, 64, 2, 16
    rows = _rand(n, (hq + 2) * d, dt=torch.bfloat16, seed=1)
    prep = types.SimpleNamespace(query_scale=None, norm_span="head", rotation=None, norm_weight_q=None, norm_weight_k=None, norm_eps=1e-5,
                                 norm_first=True)
    slots = torch.randperm(n + 11, generator=torch.Generator().manual_seed(2))[:n].int().to(DEV)
    positions = torch.arange(n, dtype=torch.int32, device=DEV)
    got = []
    for cuts in ((0, n), (0, 1 << 19, n)):
        pages = torch.zeros(n // ps + 2, 2, 1, ps, d, dtype=torch.bfloat16, device=DEV)
        q = torch.cat([ops.heads_prepare(rows[a:b], hq, 1, 1, d, d, d, prep, positions[a:b], pages, slots[a:b]) for a, b in zip(cuts, cuts[1:])])
        got.append((q, pages))
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])
    assert torch.equal(ops.heads_prepare(rows, hq, 1, 1, d, d, d, prep, positions, None, None), got[0][0])
    values = got[0][1][:, 1].reshape(-1, d, ps)[(slots // ps).long(), :, (slots % ps).long()]
    assert torch.equal(values, rows[:, -d:])


def test_wide_tiles_of_weights_of_more_than_four_gib(ops, monkeypatch):
    """A group's matrix past 2^32 bytes goes to the tiles where the rule says so, plain and with the gate, and gives the passes' bits."""
    k, nout, m = 4096, (1 << 19) + 32, 70
    w = torch.empty(1, nout, k, dtype=torch.bfloat16, device=DEV)
    w.normal_(std=0.02, generator=torch.Generator(DEV).manual_seed(1))
    x = _rand(m, k, dt=torch.bfloat16, seed=2)
    off = torch.tensor([0, m], dtype=torch.int32, device=DEV)
    took, call = [], ops._call
    monkeypatch.setattr(ops, "_call", lambda name, *a: (took.append(a[13]), call(name, *a))[1])
    monkeypatch.setattr(ops, "stream_cuts", lambda *a: (0, 1))
    for swiglu in (False, True):
        got = []
        for half, wide in ((False, False), (False, True)) + (() if swiglu else ((True, False),)):
            monkeypatch.setattr(ops, "stream_half", lambda *a: half)
            monkeypatch.setattr(ops, "stream_wide", lambda *a: wide)
            got.append(ops.gemm_stream(x, w, offsets=off, swiglu=swiglu, rows=m))
        assert all(torch.equal(g, got[0]) for g in got[1:]) and got[0].isfinite().all() and got[0][-1, -16:].any()
    assert took == [0, 1, 2, 0, 1]
