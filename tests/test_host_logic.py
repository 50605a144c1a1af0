"""Host-side rules that need no GPU: how the products split their work, the row order of a rotary weight, and how
parts take their tensors from the loader."""
from types import SimpleNamespace

import numpy as np
import pytest
import torch

from microllm_rocm_amd.architectures.qwen2 import build_spec, init_rules
from microllm_rocm_amd.ops import kernels
from microllm_rocm_amd.parts import Model, Runtime
from microllm_rocm_amd.parts.linear import MEDIUM_GATED_ROWS, MEDIUM_ROWS, SKINNY_ROWS, Weight, takes_packed, takes_unscaled
from microllm_rocm_amd.weights.random_init import random_tensors
from tiny import TINY_A, TINY_B


@pytest.mark.parametrize("n,k", [(4608, 3584), (3584, 18944), (37888, 3584), (152064, 3584), (256, 64), (896, 4864), (8192, 29568), (331, 120)])
def test_medium_plan_depends_on_the_weight_alone_and_is_launchable(n, k):
    tiles, waves, splits = kernels.medium_plan(n, k)
    assert tiles in (1, 2) and waves == 8
    assert 1 <= splits <= 16 and splits & (splits - 1) == 0
    assert splits <= max(1, -(-k // 256)), "a split takes at least one stage of 256"
    assert kernels.medium_plan(n, k, may_split=False)[2] == 1
    groups = -(-(-(-n // 16)) // (8 * tiles))
    if splits > 1:
        assert groups * (splits // 2) < kernels.MEDIUM_WORKGROUPS, "no more splits than the GPU needs"


@pytest.mark.parametrize("m,n,k,parts", [
    (2048, 3584, 18944, 2), (1024, 3584, 18944, 4), (512, 3584, 18944, 8), (65, 3584, 18944, 8),     # a long reduction into a narrow result
    (4096, 3584, 18944, 4), (8192, 3584, 18944, 4),                                                   # a last round of tiles that is not full
    (2048, 3584, 3584, 1), (2048, 4608, 3584, 1), (512, 3584, 3584, 1),                               # short reductions stay whole
    (2048, 8192, 29568, 1), (4096, 8192, 29568, 1), (512, 8192, 29568, 2), (256, 8192, 8192, 4),      # wide results fill the GPU by themselves
    (2048, 896, 4864, 2), (8192, 896, 4864, 1), (100, 331, 120, 1), (300, 64, 4160, 2), (300, 64, 4128, 1)])
def test_library_splits(m, n, k, parts):
    assert kernels.library_splits(m, n, k) == parts
    assert k % parts == 0 and (parts == 1 or k // parts >= kernels.LIBRARY_SPLIT_LENGTH)


@pytest.mark.parametrize("m,n,k,splits", [(512, 3584, 3584, 4), (512, 3584, 18944, 8), (2048, 3584, 18944, 2), (2048, 37888, 3584, 1),
                                          (300, 64, 512, 1), (100, 8192, 8192, 4), (4096, 8192, 29568, 1)])
def test_tiled_splits(m, n, k, splits):
    assert kernels.tiled_splits(m, n, k) == splits
    assert -(-k // 64) // splits >= (kernels.TILED_SPLIT_STAGES if splits > 1 else 0)


@pytest.mark.parametrize("tokens,kv_heads,longest,splits", [(1, 4, 4096, 8), (8, 4, 4096, 4), (64, 4, 4096, 1), (32, 4, 16384, 2),
                                                            (16, 4, 4096, 4), (1, 2, 300, 1), (1, 1, 100000, 195), (3, 8, 1024, 2)])
def test_decode_splits(tokens, kv_heads, longest, splits):
    assert kernels.decode_splits(tokens, kv_heads, longest) == splits


def test_query_tiles_go_in_twos_that_walk_about_as_many_keys():
    # one prompt of 2048 tokens from position 0 (16 tiles), a portion of 300 from position 1000, one tile alone
    tiles = [(0, offset, 128, offset) for offset in range(0, 2048, 128)]
    tiles += [(1, 2048 + offset, min(128, 300 - offset), 1000 + offset) for offset in range(0, 300, 128)] + [(2, 2348, 17, 40)]
    pairs = kernels.pair_query_tiles(list(tiles))
    covered = sorted((r, first, count) for r, a, ca, b, cb in pairs for first, count in ((a, ca), (b, cb)) if count)
    assert covered == sorted(tile[:3] for tile in tiles), "every tile once"
    of_first = [pair for pair in pairs if pair[0] == 0]
    position = {tile[1]: tile[3] for tile in tiles}
    weights = [position[a] + ca + position[b] + cb for _, a, ca, b, cb in of_first]
    assert len(of_first) == 8 and max(weights) == min(weights) == 2048 + 128, "late with early: all the same"
    assert [pair for pair in pairs if pair[0] == 2] == [(2, 2348, 17, 0, 0)]
    assert sorted(pair[1:] for pair in pairs if pair[0] == 1) == [(2048 + 128, 128, 0, 0), (2048 + 256, 44, 2048, 128)]
    keys = [position[a] + ca + (position[b] + cb if cb else 0) for _, a, ca, b, cb in pairs]
    assert keys == sorted(keys, reverse=True), "the longest first"
    # under a window neighbours go together
    adjacent = kernels.pair_query_tiles(list(tiles), adjacent=True)
    walked = [max(position[a] + ca, position[b] + cb if cb else 0) for _, a, ca, b, cb in adjacent]
    assert walked == sorted(walked, reverse=True), "the longest first: of neighbours the later one's keys"
    assert sorted(pair[1:] for pair in adjacent if pair[0] == 0) == [(offset, 128, offset + 128, 128) for offset in range(0, 2048, 256)]
    assert sorted(pair[1:] for pair in adjacent if pair[0] == 1) == [(2048, 128, 2048 + 128, 128), (2048 + 256, 44, 0, 0)]


@pytest.mark.parametrize("heads,kv_heads,hd,n_freq", [(4, 2, 16, 8), (3, 1, 32, 8), (28, 4, 128, 64), (2, 0, 64, 32), (5, 5, 48, 0)])
def test_rotary_pair_order_puts_partners_side_by_side(heads, kv_heads, hd, n_freq):
    order = kernels.rotary_pair_order(heads, kv_heads, hd, n_freq).tolist()
    total = (heads + 2 * kv_heads) * hd
    assert sorted(order) == list(range(total))
    for head in range(heads + 2 * kv_heads):
        rows = [row - head * hd for row in order[head * hd:(head + 1) * hd]]
        if head < heads + kv_heads:
            for pair in range(n_freq):
                assert rows[2 * pair] == pair and rows[2 * pair + 1] == pair + n_freq
            assert rows[2 * n_freq:] == list(range(2 * n_freq, hd))
        else:
            assert rows == list(range(hd)), "value heads stay as they are"


def test_parts_take_their_tensors_out_of_the_dict_as_they_bind():
    for config in (TINY_A, TINY_B):        # A ties the head to the embedding: that table is looked up twice
        spec = build_spec(config)
        model = Model(spec, Runtime(torch.float32, torch.device("cpu")))
        tensors = random_tensors(model.tensors(), init_rules(config), 0, dtype=torch.float32)
        names = set(tensors)
        untouched = dict(tensors)
        model.bind(tensors, consume=True)
        assert not tensors, "every declared tensor was handed over"
        assert model.embedding.table is untouched["model.embed_tokens.weight"]
        if config.tie_word_embeddings:
            assert model.head.weight.tensor is model.embedding.table
        # without consume the dict is left as it was
        again = Model(spec, Runtime(torch.float32, torch.device("cpu")))
        again.bind(untouched)
        assert set(untouched) == names


def test_which_product_a_linear_takes(monkeypatch):
    plain = Weight(torch.zeros((64, 32), dtype=torch.bfloat16))          # on the host nothing is packed
    assert plain.packed is None and not takes_packed(plain, 1) and not takes_unscaled(plain, 1)
    packed = Weight(torch.zeros((64, 32), dtype=torch.bfloat16), pack=False)
    packed.packed = torch.zeros((4, 1, 4, 16, 8), dtype=torch.bfloat16)   # as on the GPU
    assert takes_packed(packed, SKINNY_ROWS) and takes_packed(packed, MEDIUM_ROWS) and not takes_packed(packed, MEDIUM_ROWS + 1)
    assert takes_packed(packed, MEDIUM_GATED_ROWS, gated=True) and not takes_packed(packed, MEDIUM_GATED_ROWS + 1, gated=True), \
        "the gated product goes to the library (and the SiLU kernel) beyond this many rows"
    assert takes_unscaled(packed, SKINNY_ROWS) and not takes_unscaled(packed, SKINNY_ROWS + 1)
    packed.tensor = None                                                   # one copy: the packed one serves every step
    assert takes_packed(packed, 5000) and takes_packed(packed, 40, gated=True)
    wide = Weight(torch.zeros((16, 8), dtype=torch.bfloat16), pack=False)
    wide.packed, wide.out_features = packed.packed, 2048 * 16
    assert takes_packed(wide, 40) and not takes_packed(wide, 41), "many tiles and a short reduction: the library's from 41 rows on"
    for reduction, taken in ((504, False), (512, True)):                    # the head of a model
        head = Weight(torch.zeros((16, reduction), dtype=torch.bfloat16), pack=False)
        head.packed, head.out_features = packed.packed, 2048 * 16
        assert takes_packed(head, 40, address=2) and takes_packed(head, 41) == takes_packed(head, 64) == taken and not takes_packed(head, 65)
        assert not takes_packed(head, 41, address=2), "rows at no 16-byte boundary are the library's"
        monkeypatch.setattr(kernels, "library_tuning", lambda: True)
        assert takes_packed(head, 40) and not takes_packed(head, 41), "and so are those of a tuned one"
        monkeypatch.undo()
        head.out_features -= 16                                              # a tile fewer
        assert takes_packed(head, 64, address=2)


def test_percentile_interpolates_between_the_two_nearest_sorted_values():
    from microllm_rocm_amd.cli.hf_infer import percentile
    assert percentile([4, 1, 3, 2], 0.5) == 2.5 and percentile([7.0], 0.95) == 7.0
    assert percentile([1, 2, 3, 4, 5], 0.95) == pytest.approx(4.8) and percentile([5, 1], 0.0) == 1 and percentile([5, 1], 1.0) == 5
    with pytest.raises(ValueError):
        percentile([], 0.5)


def test_padding_a_step_to_a_graph_shape_never_changes_the_kernel_a_product_takes():
    """A mixed step is padded to fixed numbers of token rows and of wanted rows before it is replayed from a graph;
    the padded count must take the same product as the real one, for every kind of weight, or the replayed step
    would give other bits than the same step run eagerly."""
    from microllm_rocm_amd.engine.engine import MAX_GRAPH_TOKENS, MAX_GRAPH_WANTED, _token_rows, _wanted_rows
    narrow = Weight(torch.zeros((64, 32), dtype=torch.bfloat16), pack=False)
    narrow.packed = torch.zeros((4, 1, 4, 16, 8), dtype=torch.bfloat16)
    wide = Weight(torch.zeros((16, 8), dtype=torch.bfloat16), pack=False)
    wide.packed, wide.out_features = narrow.packed, 2048 * 16

    def kernel_of(weight, rows, gated):
        return (rows <= SKINNY_ROWS, takes_unscaled(weight, rows), takes_packed(weight, rows, gated), rows <= MEDIUM_ROWS)

    for pad, most in ((_token_rows, MAX_GRAPH_TOKENS), (_wanted_rows, MAX_GRAPH_WANTED)):
        for rows in range(1, most + 1):
            padded = pad(rows)
            assert rows <= padded <= max(16, 2 * rows)
            for weight in (narrow, wide):
                for gated in (False, True):
                    assert kernel_of(weight, rows, gated) == kernel_of(weight, padded, gated), (pad.__name__, rows, padded)


def test_kept_graphs_stay_bounded_and_mixed_shapes_never_push_decode_graphs_out():
    """More recurring shapes than the budget holds: captures stay bounded (a shape that was captured and evicted
    twice runs eagerly from then on), decode graphs are not evicted by mixed ones, and both budgets hold in bytes."""
    from types import SimpleNamespace
    from microllm_rocm_amd.engine.graphs import MAX_CAPTURES_A_SHAPE, GraphPolicy
    policy = GraphPolicy(decode_graphs=4, mixed_graphs=3, most_bytes=1000, seen_before_capture=2)
    captures = 0
    for key in range(4):                                   # four decode shapes, captured once each
        policy.decode.put(("decode", key), SimpleNamespace(held_bytes=100))
    assert len(policy.decode) == 4
    shapes = [("mixed", index) for index in range(10)]      # ten mixed shapes that keep coming round
    for round_number in range(40):
        for key in shapes:
            if not policy.wants_mixed(key):
                continue
            if policy.mixed.get(key) is None:
                state = SimpleNamespace(held_bytes=0)
                policy.mixed.put(key, state, policy.evicted_mixed)
                state.held_bytes = 100                      # the capture
                captures += 1
                policy.captured_mixed(key)
                policy.mixed.trim(policy.evicted_mixed, keep=key)
            assert len(policy.mixed) <= 3 and policy.mixed.held_bytes() <= 500
    assert captures <= MAX_CAPTURES_A_SHAPE * len(shapes), "no shape is captured over and over"
    assert len(policy.decode) == 4 and all(("decode", key) in policy.decode for key in range(4))
    assert all(not policy.wants_mixed(key) or key in policy.mixed for key in shapes), "evicted twice: eagerly for good"
    # a shape seen once is not captured; the second time it is
    fresh = GraphPolicy(seen_before_capture=2)
    assert not fresh.wants_mixed("s") and fresh.wants_mixed("s")
    # the budget in bytes: a graph of large logits pushes older ones out, the one in use stays
    small = GraphPolicy(decode_graphs=8, mixed_graphs=8, most_bytes=600)
    for key in range(3):
        small.decode.put(key, SimpleNamespace(held_bytes=100))
    small.decode.put("large", SimpleNamespace(held_bytes=250))
    assert "large" in small.decode and small.decode.held_bytes() <= 300 and 0 not in small.decode


# 16 splits from 8192 positions on, 8 below: of a step planned for 4096 the keys are often little more than half, and 16 were slower than the 8 of before
@pytest.mark.parametrize("tokens,kv_heads,longest,head_dim,splits", [
    (1, 4, 1023, 128, 1), (1, 4, 1024, 128, 8), (1, 4, 4096, 128, 8), (1, 4, 8191, 128, 15), (4, 4, 4096, 128, 8), (4, 4, 8191, 128, 15), (4, 4, 8192, 128, 16),
    (8, 2, 4096, 64, 8), (1, 4, 32768, 128, 32), (8, 4, 4096, 128, 8), (16, 4, 1024, 128, 4), (17, 4, 1024, 128, 2), (32, 4, 1024, 128, 1), (64, 4, 4096, 128, 1),
    (32, 2, 1024, 64, 4), (1, 1, 511, 256, 1), (1, 1, 512, 256, 4), (32, 1, 512, 256, 4), (33, 1, 512, 256, 1), (33, 1, 1023, 256, 1), (64, 1, 1024, 256, 4),
    (2, 1, 2048, 256, 16), (8, 1, 4096, 256, 16), (1, 1, 100000, 128, 195), (0, 1, 0, 64, 1)])
def test_decode_parts(tokens, kv_heads, longest, head_dim, splits):
    assert kernels.decode_parts(tokens, kv_heads, longest, head_dim) == splits
    assert splits >= kernels.decode_splits(tokens, kv_heads, longest)


def test_tiles_of_half_the_queries_where_whole_ones_leave_compute_units_idle():
    from microllm_rocm_amd.parts.attention import QueryTilePlanner
    assert QueryTilePlanner(False).tile_rows([512]) == [128]
    planner = QueryTilePlanner(False, 14)
    assert planner.tile_rows([]) == []
    # 9 pairs of tiles of 14 heads: 126; a portion of one tile has one workgroup either way
    assert [planner.tile_rows([count])[0] for count in (2, 128, 129, 2048, 2304, 2305)] == [128, 128, 64, 64, 64, 128]
    assert planner.tile_rows([512, 128, 600]) == [64, 128, 64] and planner.tile_rows([300] * 5) == [128] * 5
    assert planner.key != QueryTilePlanner(False, 28).key


def test_neighbouring_tiles_share_a_workgroup_where_a_step_has_more_than_a_round_of_them():
    from microllm_rocm_amd.parts.attention import QueryTilePlanner
    planner = QueryTilePlanner(False, 28)       # 9 workgroups a head: 252, 10: 280
    assert [planner.neighbours(counts) for counts in ([2304], [2305], [1, 2303], [128] * 9, [128] * 10, [])] == [False, True, True, False, True, False]
    small = QueryTilePlanner(False, 28, 32)     # two workgroups a unit: 18 a head, 504, and 19, 532
    assert [small.neighbours([count]) for count in (2305, 4608, 4609)] == [False, False, True] and small.key != planner.key
    assert QueryTilePlanner(False, 28, 48).key == planner.key
    assert not QueryTilePlanner(False).neighbours([100000]) and QueryTilePlanner(True).neighbours([2])
    host = SimpleNamespace(counts=[2305], cu=[0, 2305], starts=[0], totals=[2305], single_tokens_only=False)
    tiles = planner.plan(host)[0]["tiles"]
    assert tiles[0].tolist() == [0, 2304, 1, 0, 0] and tiles[1].tolist() == [0, 2048, 128, 2176, 128]
    assert sorted(tiles[:, 2] + tiles[:, 4]) == [1] + [256] * 9
    assert [max(a + ca, b + cb) for _, a, ca, b, cb in tiles.tolist()] == [2305] + list(range(2304, 0, -256)), "by the keys they walk"


@pytest.mark.parametrize("tokens,heads,kv_heads,head_dim,chunks,dtype,splits", [
    (73, 28, 4, 128, 200, torch.float32, True), (74, 28, 4, 128, 8, torch.float32, True), (292, 28, 4, 128, 8, torch.float32, True),
    (293, 28, 4, 128, 8, torch.float32, False), (292, 28, 4, 128, 64, torch.float32, False), (292, 28, 4, 120, 8, torch.float32, False),
    (127, 32, 8, 128, 8, torch.float32, True), (128, 32, 8, 128, 8, torch.float32, False), (256, 8, 8, 128, 8, torch.float32, False),
    (74, 28, 4, 128, 8, torch.bfloat16, False), (74, 28, 4, 144, 8, torch.float32, False)])
def test_rowwise_splits(tokens, heads, kv_heads, head_dim, chunks, dtype, splits):
    assert kernels.rowwise_splits(tokens, heads, kv_heads, head_dim, chunks, dtype) == splits


@pytest.mark.parametrize("tokens,heads,kv_heads,requests,keys,splits", [
    (80, 28, 4, 2, 48, False), (80, 28, 4, 2, 49, True), (80, 32, 8, 2, 64, False), (80, 32, 8, 2, 65, True), (80, 28, 4, 80, 24, False),
    (80, 28, 4, 80, 25, True), (73, 28, 4, 2, 10, True), (80, 28, 4, 0, 0, True)])
def test_rowwise_splits_of_few_keys(tokens, heads, kv_heads, requests, keys, splits):
    """Rows of few keys stay with a wave a row, from as many rows on as may have one."""
    assert kernels.rowwise_splits(tokens, heads, kv_heads, 128, 2, torch.float32, requests, keys) == splits
