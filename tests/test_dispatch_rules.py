"""Which calls the kernels' dispatch lets through, without a GPU."""
import types

import pytest
import torch

from jax_llm_examples_amd.ops.hip import HipOps


def tensor(rows, cols, device="cuda:0", dtype=torch.float32):
    """What the rule looks at of a matrix on a GPU."""
    return types.SimpleNamespace(dtype=dtype, shape=(rows, cols), dim=lambda: 2,
                                 get_device=lambda: int(device[5:]) if device.startswith("cuda") else -1, is_contiguous=lambda: True, data_ptr=lambda: 4096)


def rule(h, w, act=-1):
    ops = types.SimpleNamespace(gemm_f32_rows=lambda *a: "rows", gemm_f32_split=lambda *a: "split", _compute_units=256, _device_index=0,
                                split_ranges=HipOps.split_ranges)
    return HipOps._dense_float32(ops, h, w, act)


def test_dense_float32_products_by_size():
    assert rule(tensor(1, 64), tensor(32, 64)) == "rows"
    assert rule(tensor(512, 4096), tensor(4096, 4096)) == "split"
    assert rule(tensor(512, 4096, dtype=torch.bfloat16), tensor(4096, 4096)) is None
    assert rule(tensor(1, 64), tensor(32, 60)) is None  # (the library's product refuses it)


@pytest.mark.parametrize("rows, n, k, gated, pays", [(9, 64, 64, False, True), (128, 64, 64, False, True), (129, 64, 64, False, False),
    (32, 2048, 2048, False, True), (33, 2048, 2048, False, False), (64, 1024, 1024, False, True), (65, 1024, 1024, False, False), (128, 2048, 512, False, False),
    (64, 2048, 2048, True, True), (65, 2048, 2048, True, False), (16, 512, 2052, False, False),
    (64, 32, 2048, False, False), (64, 32, 2048, True, False), (32, 1535, 2048, False, False), (32, 1536, 2048, False, True),
    (16, 2046, 2048, True, False), (16, 2048, 2048, True, True), (64, 32, 1024, False, True), (9, 32, 1028, False, False),
    (16, 512, 508, False, False), (16, 512, 512, False, True), (16, 511, 64, False, True), (17, 512, 128, False, True),
    (17, 512, 124, False, False), (16, 512, 64, True, True)])
def test_dense_float32_products_of_tens_of_rows_by_size(rows, n, k, gated, pays):
    assert HipOps.f32_tiles_pay(rows, n, k, gated) == pays


@pytest.mark.parametrize("units", [32, 64, 128, 256])
def test_dense_float32_products_of_tens_of_rows_are_one_round_of_any_device(units):
    """A device with fewer compute units, as a part of one has: as many blocks are several rounds of it."""
    assert HipOps.f32_tiles_pay(16, 32 * units, 1024, True, units) and not HipOps.f32_tiles_pay(16, 32 * units + 32, 1024, True, units)
    assert HipOps.f32_tiles_pay(48, 32 * (units // 3), 512, True, units) and not HipOps.f32_tiles_pay(49, 32 * (units // 3), 512, True, units)


@pytest.mark.parametrize("rows", [1, 512])
@pytest.mark.parametrize("a, b", [("cuda:0", "cuda:1"), ("cuda:1", "cuda:0"), ("cuda:0", "cpu"), ("cpu", "cuda:0"),
                                  ("cuda:1", "cuda:1")])
def test_matrices_elsewhere_are_left_to_the_library(rows, a, b):
    assert rule(tensor(rows, 4096, a), tensor(4096, 4096, b)) is None


def test_leave_for_shared_memory_is_asked_for_on_the_device_of_the_launch():
    """What a kernel may use of a compute unit's shared memory is an attribute of a device: a process with two must not
    remember the first one's.  (One place asks for it, and no launcher keeps an answer.)"""
    import glob
    import os
    from jax_llm_examples_amd.ops import build
    asks = []
    for path in glob.glob(os.path.join(build.CSRC, "*.h*")):
        with open(path) as f:
            for line in f:
                if "hipFuncSetAttribute" in line:
                    asks.append(os.path.basename(path))
                kept = line.strip().startswith("static ") and ("allowed" in line or "hipError_t" in line)
                assert not kept, (path, line)
    assert asks == ["common.h"]


@pytest.mark.parametrize("requests, tokens, behind, heads, rank, formed", [
    (1, 2048, 0, 32, 512, True), (64, 20, 0, 32, 512, True), (1, 512, 8192, 32, 512, True), (64, 24, 168, 32, 512, True),
    (1, 2048, 0, 8, 256, True), (2, 954, 0, 8, 512, True),
    (200, 8, 56, 16, 512, False), (200, 8, 56, 32, 512, False), (128, 16, 112, 32, 512, False),  # many short portions
    (1, 64, 8192, 16, 512, False), (8, 1, 2000, 16, 512, False), (1, 128, 8192, 16, 512, False),
    (1, 186, 4000, 2, 512, False), (1, 174, 8000, 1, 64, False), (1, 463, 8000, 1, 128, False),  # few heads: one long chain
    (1, 88, 500, 32, 64, False), (2, 8, 0, 2, 256, False)])
def test_which_steps_form_keys_and_values(requests, tokens, behind, heads, rank, formed):
    segments = [tokens] * requests, [behind] * requests, 0
    _, blocks, rows, pairs = HipOps.expanded_plan(*segments)
    assert HipOps.expansion_pays(requests * tokens, heads, rank, rows, pairs, len(blocks) // 4,
                                 HipOps.expanded_steps(*segments)) == formed


@pytest.mark.parametrize("window", [0, 1, 63, 64, 500])
def test_the_longest_block_of_a_step(window):
    lens, starts = [1, 64, 129, 700, 5], [0, 63, 128, 1000, 777]
    for one in [*zip(lens, starts), None]:
        ln, st = ([one[0]], [one[1]]) if one else (lens, starts)
        blocks, keys = HipOps.expanded_plan(ln, st, window)[1], []
        for n0, nt in zip(blocks[::4], blocks[1::4]):
            seg = next(i for i in range(len(ln)) if sum(ln[: i + 1]) > n0)
            pos = st[seg] + n0 - sum(ln[:seg])
            first = max(0, pos - window + 1) if window else 0
            keys.append((pos + nt - 1) // 64 - first // 64 + 1)
        assert max(keys) - 2 <= HipOps.expanded_steps(ln, st, window) <= max(keys)


@pytest.mark.parametrize("groups, rows, blocks, wide", [(8, 410, 56, True), (16, 410, 64, True), (8, 192, 56, True), (8, 170, 56, False),
                                                        (2, 300, 32, False), (4, 300, 16, False), (4, 410, 56, False)])
def test_few_groups_stay_with_passes(groups, rows, blocks, wide):
    """Of few groups one may be far fuller than the others, and is then what the launch takes: it is cut in more pieces."""
    assert HipOps.stream_wide(rows * groups, groups, blocks) == wide


@pytest.mark.parametrize("groups, rows, blocks, wide", [(64, 290, 2, False), (32, 330, 2, False), (24, 290, 4, False), (64, 192, 4, False), (128, 176, 3, False),
                                                        (16, 300, 20, True), (8, 410, 16, True), (16, 700, 64, True), (10, 384, 12, False), (16, 512, 20, True), (16, 160, 64, False)])
def test_wide_tiles_where_their_row_blocks_reach_every_chiplet(groups, rows, blocks, wide):
    """Few row blocks of wide tiles are on a few of the eight chiplets only, where passes are dealt to all of them."""
    assert HipOps.stream_wide(rows * groups, groups, blocks) == wide


@pytest.mark.parametrize("groups, rows, blocks, half", [
    (8, 512, 32, False), (8, 512, 16, False), (8, 410, 32, False), (8, 190, 32, False), (8, 330, 32, False), (8, 128, 32, False),
    (8, 64, 32, False), (8, 64, 16, False), (16, 128, 40, False), (16, 256, 40, False), (4, 512, 16, False), (8, 700, 16, False),
    (8, 128, 16, True), (8, 300, 16, True), (8, 512, 8, True), (16, 160, 8, True), (8, 160, 24, True), (64, 190, 2, False)])
def test_narrower_tiles_where_wide_ones_leave_compute_units_idle(groups, rows, blocks, half):
    assert HipOps.stream_half(rows * groups, groups, blocks) == half


@pytest.mark.parametrize("groups", [8, 10, 12, 16, 20, 24])
def test_narrower_tiles_are_one_round_however_the_rows_are_shared_out(groups):
    """The tiles of a group as the kernel cuts them, its row blocks dealt to the eight chiplets in turn: none gets more than
    its 32 compute units, with even groups, uneven ones, from 0.3 to 1.7 of the mean, and 40 % of the rows in one."""
    g = torch.Generator().manual_seed(groups)
    taken = 0
    for blocks in range(1, 49):
        for mean in range(90, 900, 20):
            if not HipOps.stream_half(mean * groups, groups, blocks):
                continue
            taken += 1
            weight = torch.exp(0.25 * torch.randn(groups, generator=g))
            for part in (torch.ones(groups), weight, torch.linspace(0.3, 1.7, groups), torch.tensor([0.4 * groups] + [0.6 * groups / (groups - 1)] * (groups - 1))):
                rows = (part / part.sum() * mean * groups).int()
                assert -(-blocks // 8) * int(((rows + 287) // 288).sum()) <= 32, (blocks, mean, rows.tolist())
    assert taken


@pytest.mark.parametrize("rows, groups, blocks, k, units, cut", [
    (64, 1, 125, 4096, 256, (125, 2)), (64, 1, 196, 4096, 256, (0, 1)), (64, 1, 256, 4096, 256, (0, 1)), (64, 1, 257, 4096, 256, (1, 4)),
    (192, 1, 790, 5120, 256, (22, 5)), (193, 1, 790, 5120, 256, (0, 1)), (64, 1, 125, 4032, 256, (0, 1)), (64, 1, 125, 4096, 64, (0, 1)),
    (64, 1, 80, 4096, 64, (16, 4)), (64, 1, 125, 4096, 1, (0, 1)), (16 * 128, 16, 20, 8192, 256, (4, 4)), (16 * 172, 16, 20, 8192, 256, (4, 4)), (16 * 173, 16, 20, 8192, 256, (0, 1)),
    (16 * 128, 16, 64, 5120, 256, (0, 1)), (8 * 64, 8, 16, 7168, 256, (16, 2)), (8 * 64, 8, 8, 4096, 256, (8, 4)), (3 * 64, 3, 86, 4096, 256, (1, 4)),
    (100 * 3, 100, 3, 4096, 256, (1, 2)), (0, 129, 1, 8192, 256, (0, 1))])
def test_which_blocks_of_a_product_in_passes_are_cut(rows, groups, blocks, k, units, cut):
    assert HipOps.stream_cuts(rows, groups, blocks, k, units) == cut


@pytest.mark.parametrize("groups, nout, k, rows, way", [
    (8, 1024, 8192, 128, "cut"), (8, 1024, 8192, 96, "cut"), (8, 1024, 8192, 192, "tiles"), (8, 1024, 4096, 160, "cut"), (16, 512, 4096, 128, "cut"),
    (8, 2048, 4096, 128, "tiles"), (8, 2048, 5120, 128, "tiles"), (8, 2048, 6144, 128, "cut"), (16, 1024, 8192, 128, "cut"), (16, 1024, 4096, 128, "tiles"),
    (8, 1536, 4096, 160, "tiles"), (8, 1536, 8192, 160, "cut"), (8, 3072, 8192, 160, "tiles"), (24, 1024, 8192, 128, "tiles"), (8, 2048, 2048, 128, "tiles"),
    (8, 14336, 4096, 410, "wide"), (8, 4096, 7168, 48, "cut"), (8, 4096, 2048, 64, "whole")])
def test_plain_products_of_groups_by_size(monkeypatch, groups, nout, k, rows, way):
    """Of passes, passes cut along k and the two kinds of tiles the one that a call of drawn groups launches."""
    called = []
    ops = types.SimpleNamespace(_compute_units=256, _chk=lambda *a: None, stream_supported=lambda *a: True, _query=lambda *a: 1,
                                _call=lambda name, *a: called.append((a[13], a[16])))
    for rule_ in ("stream_half", "stream_wide", "stream_cuts", "cut_passes_pay"):
        setattr(ops, rule_, getattr(HipOps, rule_, lambda *a: False))
    a = torch.empty(1, dtype=torch.bfloat16).expand(groups * rows, k)
    b = torch.empty(1, dtype=torch.bfloat16).expand(groups, nout, k)
    monkeypatch.setattr(torch, "empty", lambda *a, **kw: None)
    HipOps.gemm_stream(ops, a, b, offsets=torch.zeros(groups + 1, dtype=torch.int32))
    assert called == [{"wide": (1, 1), "tiles": (2, 1), "whole": (0, 1), "cut": (0, HipOps.stream_cuts(groups * rows, groups, -(-nout // 256), k, 256)[1])}[way]]
    assert (called[0][1] > 1) == (way == "cut")


@pytest.mark.parametrize("n, k, least, most", [(16000, 2048, 5, 64), (28672, 4096, 5, 64), (28688, 4096, 5, 32), (32768, 2048, 5, 32),
                                                 (32784, 2048, 5, 16), (50000, 3072, 5, 16), (65536, 4096, 5, 24), (202048, 5120, 5, 24)])
def test_output_heads_by_size(n, k, least, most):
    """In the streaming layout, where that layout has no kernel of its own for many rows, and row-major."""
    few = lambda tiled, streams: [r for r in range(1, 130) if HipOps.head_few(r, n, k, tiled, streams)]
    assert few(True, True) == list(range(least, most + 1))
    assert few(True, False) == list(range(least, 65))
    assert few(False, False) == list(range(1, 65))


@pytest.mark.parametrize("k, rows, groups, swiglu, pays", [
    (2048, 16, 8, True, True), (1088, 128, 64, False, True), (1024, 16, 32, True, False), (768, 128, 128, False, False),
    (1024, 2, 16, False, True), (1024, 2, 16, True, False), (1024, 3, 16, False, False), (1024, 96, 8, True, True), (1024, 95, 8, True, False),
    (64, 1, 4, False, True)])
def test_short_rows_of_weights_stay_with_the_weight_streaming_product(k, rows, groups, swiglu, pays):
    assert HipOps.few_pays(k, rows, groups, swiglu) == pays


@pytest.mark.parametrize("k, rows, last, product", [(2048, 4, False, "few"), (1024, 4, False, "skinny"), (1024, 2, False, "few"),
                                                     (1024, 48, False, "few"), (1024, 48, True, "skinny"), (72, 4, False, "skinny")])
def test_experts_products_go_where_they_pay(k, rows, last, product):
    """Four groups, and with the shared expert's one more; rows that are picked count, not those they are picked from."""
    at = lambda *shape: types.SimpleNamespace(dtype=torch.bfloat16, shape=shape, data_ptr=lambda: 4096, numel=lambda: shape[0] * shape[1])
    ops = types.SimpleNamespace(gemm_few=lambda *a, **kw: "few", gemm_skinny=lambda *a, **kw: "skinny", few_pays=HipOps.few_pays)
    ops._few_fits = lambda *a: HipOps._few_fits(ops, *a)
    b, more = at(4, 256, k), dict(b_last=at(256, k)) if last else {}
    assert HipOps._few_experts(ops, at(rows, k), b, **more) == product
    assert HipOps._few_experts(ops, at(200, k), b, a_rows=types.SimpleNamespace(numel=lambda: rows), **more) == product
    assert HipOps._few_experts(ops, at(200, k), b, a_rows=types.SimpleNamespace(numel=lambda: 999), rows=rows, **more) == product


@pytest.mark.parametrize("lens, heads, dk, dv, pays", [
    ([64], 16, 128, 128, False), ([256], 16, 128, 128, True), ([2048], 4, 64, 64, True), ([64] * 32, 16, 128, 128, True),
    ([80] * 25, 16, 128, 128, True), ([32] * 64, 16, 128, 128, False), ([36] * 64, 64, 128, 128, False),
    ([65] * 32, 16, 128, 128, False), ([32] * 128, 16, 64, 64, False), ([65] * 32, 32, 64, 128, False),
    ([80] * 16, 32, 64, 128, False), ([36, 51, 53] * 20, 2, 128, 16, False), ([80] * 16, 8, 128, 256, True)])
def test_which_segments_go_by_chunks(lens, heads, dk, dv, pays):
    """A chunk of 64 places costs the same however many are filled: segments that fill theirs poorly stay with the scan."""
    assert HipOps.delta_chunks_pay(lens, heads, dk, dv) == pays


def test_few_rows_of_float32():
    assert [rule(tensor(8, 2048), tensor(n, 2048)) for n in (2048, 8192)] == ["rows", None]
    assert [rule(tensor(8, 4096), tensor(4096, 4096), act) for act in (-1, 0)] == [None, "rows"]
    assert rule(tensor(5, 8192), tensor(2048, 8192)) == rule(tensor(4, 4096), tensor(14336, 4096)) == "rows"


def test_many_rows_of_float32_with_a_short_k():
    sizes = [(777, 16384, 96), (2048, 5120, 96), (777, 16384, 2048), (1554, 2048, 8192), (512, 4096, 4096)]
    assert [HipOps.split_ranges(*s, False, 256) > 0 for s in sizes] == [False, False, True, True, True]
    assert HipOps.split_ranges(1024, 7168, 96, True, 256) == 1  # (the activation is a pass of its own behind the library's)


@pytest.mark.parametrize("n, d, experts, one", [(1, 2048, 10, True), (1, 1032, 10, True), (1, 1032, 11, False), (15, 512, 16, False), (16, 512, 16, True),
                                                (16, 2048, 16, True), (15, 2460, 10, False), (256, 2560, 16, True), (257, 64, 2, False), (1, 62, 2, False)])
def test_logits_and_choice_in_one_launch_by_size(n, d, experts, one):
    assert HipOps.choose_by_token(n, d, experts) == one


@pytest.mark.parametrize("d, experts, top_k, rows", [(2048, 10, 2, 32), (4096, 16, 1, 64), (4104, 16, 1, 16), (8192, 8, 2, 32), (8192, 9, 2, 16),
                                                     (2048, 17, 1, 16), (2048, 16, 8, 16)])
def test_rows_normed_and_chosen_for_in_one_launch(d, experts, top_k, rows):
    assert HipOps.norm_choose_rows(d, experts, top_k) == rows


@pytest.mark.parametrize("rows, n, k, tile", [
    (2048, 4096, 4096, (8, 4)), (2048, 5120, 5120, (8, 5)), (2048, 7168, 5120, (8, 7)), (2048, 4096, 512, (4, 4)),
    (8191, 4096, 4096, None), (4096, 8192, 2048, None), (704, 4096, 7168, None), (1024, 2048, 8192, None),
    (65, 2048, 2048, None), (192, 2048, 2048, (4, 4)),
    (2048, 4096, 4100, None), (2048, 4100, 4096, None), (0, 4096, 4096, None), (2048, 0, 4096, None), (2048, 4096, 0, None)])
def test_dense_products_of_many_rows_by_size(rows, n, k, tile):
    assert HipOps.dense_tile(rows, n, k) == (0 if tile is None else tile[0] * 16 + tile[1])


def test_dense_products_that_are_left_to_the_library():
    """Matrices elsewhere, of other types, strides and addresses, calls that derivatives are taken of."""
    def at(rows, cols, **other):
        of = dict(dtype=torch.bfloat16, shape=(rows, cols), dim=lambda: 2, get_device=lambda: 0, is_contiguous=lambda: True, data_ptr=lambda: 4096,
                  requires_grad=False)
        return types.SimpleNamespace(**{**of, **other})

    ops = types.SimpleNamespace(_compute_units=256, _device_index=0, gemm_dense=lambda h, w, tile, bias: tile)
    h, w = at(2048, 4096), at(4096, 4096)
    taken = lambda *a, **kw: HipOps._dense(ops, *a, **kw) is not None
    assert taken(h, w) and not taken(h, at(4096, 4032))
    for other in (dict(dtype=torch.float32), dict(dim=lambda: 3), dict(get_device=lambda: 1), dict(get_device=lambda: -1),
                  dict(is_contiguous=lambda: False), dict(data_ptr=lambda: 4104), dict(requires_grad=True)):
        assert not taken(at(2048, 4096, **other), w) and not taken(h, at(4096, 4096, **other))
    bias = torch.zeros(4096, dtype=torch.bfloat16)
    assert not taken(h, w, bias=bias)  # (on the CPU)
    with torch.autograd.forward_ad.dual_level():
        assert not taken(h, w)
    with torch.no_grad():
        assert taken(at(2048, 4096, requires_grad=True), w)


class Elsewhere(torch.Tensor):
    """A class of its own around no memory, whose operations it answers itself."""
    __torch_function__ = torch._C._disabled_torch_function_impl

    @staticmethod
    def __new__(cls, rows, cols):
        return torch.Tensor._make_wrapper_subclass(cls, (rows, cols), dtype=torch.bfloat16, device="cuda:0")

    @classmethod
    def __torch_dispatch__(cls, func, types, args=(), kwargs=None):
        return func


def test_dense_products_that_others_look_into_are_left_to_the_library():
    def at(rows, cols, address=4096):
        return types.SimpleNamespace(dtype=torch.bfloat16, shape=(rows, cols), dim=lambda: 2, get_device=lambda: 0, is_contiguous=lambda: True,
                                     data_ptr=lambda: address, requires_grad=False)

    ops = types.SimpleNamespace(_compute_units=256, _device_index=0, gemm_dense=lambda h, w, tile, bias: tile)
    h, w = at(2048, 4096), at(4096, 4096)
    taken = lambda h=h, w=w, **kw: HipOps._dense(ops, h, w, **kw) is not None
    assert taken() and not taken(h=Elsewhere(2048, 4096)) and not taken(w=Elsewhere(4096, 4096)) and not taken(h=at(2048, 4096, address=0))

    class Mode(torch.overrides.TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    with Mode():
        assert not taken()
    with torch.device("cpu"):
        assert taken()
        with Mode():
            assert not taken()
    try:
        torch.set_autocast_enabled("cuda", True)
        assert not taken()
    finally:
        torch.set_autocast_enabled("cuda", False)
    seen = []
    torch.jit.trace(lambda x: (seen.append(taken()), x)[1], torch.zeros(1), check_trace=False)
    assert seen and not any(seen) and taken()
