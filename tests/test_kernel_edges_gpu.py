"""The kernels at the sizes where their tiles, their remainders and the choice between them can go wrong."""
import ctypes
import math

import numpy as np
import pytest
import torch

from test_kernels_gpu import DEVICE, build_paged_case, kernels, key_page_shape, query_tile_list, reference_attention, to_bf16_exact, tolerance, value_page_shape

from microllm_rocm_amd.ops import library

pytestmark = pytest.mark.gpu

F32_STEP = 2.0 ** -24       # half a unit in the last place, relative


def device(values, dtype=torch.float32):
    return torch.as_tensor(np.asarray(values)).to(dtype).to(DEVICE)


# 128 | 129 tiles (half ones below), 288, 512, 521, 768 | 769 (two a workgroup above, at 16 rows from 521 or 768 on), 1024, 2048
@pytest.mark.parametrize("n", [16, 2048, 2049, 2064, 4608, 8192, 8336, 12288, 12304, 16384, 16400, 32768])
@pytest.mark.parametrize("k", [8, 32, 480, 544, 1536, 4128])
def test_streaming_product_tiles(n, k):
    """Any float32 sum of exact bfloat16 products errs by at most k roundings of the sum of their sizes; a row's bits are the
    same in every batch."""
    rng = np.random.default_rng(n + k)
    x_exact, x = to_bf16_exact(rng.normal(size=(64, k)))
    w_exact, w = to_bf16_exact(rng.normal(size=(n, k)))
    packed = kernels().pack_weight(w)
    whole = kernels().gemm_skinny(x, packed, n, "f32")
    bound = (k + 1) * F32_STEP * (np.abs(x_exact) @ np.abs(w_exact).T)
    assert (np.abs(whole.double().cpu().numpy() - x_exact @ w_exact.T) <= bound).all()
    for m in (1, 4, 5, 8, 9, 16, 17, 33, 48):
        assert torch.equal(kernels().gemm_skinny(x[:m].contiguous(), packed, n, "f32"), whole[:m]), m


@pytest.mark.parametrize("n,k", [(331, 120), (896, 901), (4096, 64), (1000, 1536), (6150, 700), (65560, 640), (37888, 64)])
def test_float32_product_has_one_order_of_sums_in_every_kernel(n, k):
    """The vector kernels, that of few rows (one and two tiles a wave, up to 16 and 32 rows, several groups of them), tiles of four
    shapes and small tiles for few workgroups: each element is the chain of fused multiply-adds in ascending k, so every batch gives
    a row the same bits."""
    rng = np.random.default_rng(n)
    a = device(rng.normal(size=(1003, k)))
    w = device(rng.normal(size=(n, k)))
    whole = kernels().gemm_f32(a, w)
    bound = (k + 1) * F32_STEP * (a.abs().double() @ w.abs().double().T)
    assert bool(((whole.double() - a.double() @ w.double().T).abs() <= bound).all())
    for rows in (1, 2, 5, 9, 15, 16, 17, 24, 31, 32, 33, 64, 65, 100, 127, 129, 320):
        assert torch.equal(kernels().gemm_f32(a[1003 - rows:].contiguous(), w), whole[1003 - rows:]), rows


@pytest.mark.parametrize("heads,kv_heads,hd,page_size", [(28, 4, 16, 16), (14, 2, 32, 32), (10, 2, 48, 48), (7, 1, 64, 16), (6, 3, 80, 48), (5, 1, 96, 16),
                                                         (4, 2, 112, 32), (4, 4, 128, 48)])
@pytest.mark.parametrize("broken", [None, float("inf"), float("nan")])
def test_runs_of_a_requests_tokens_have_a_tokens_bits(heads, kv_heads, hd, page_size, broken):
    """Portions that end before, on and after a stretch of 16, alone and several to a block of 16 tokens, on the kernel of stretches
    (a step that is not split, of 47 tokens a request and 58 million multiplications) and, where a block holds too many, on that of a wave a
    row; against each of the same tokens alone by a wave a chunk. A value that is not finite changes the tokens after it
    alone. Every head size of the kernel; pages of 48 positions, which tiles of 64 keys straddle."""
    rng = np.random.default_rng(hd)
    lengths, counts = [300, 16, 17, 140, 40, 5, 129, 33, 64], [290, 16, 17, 1, 2, 5, 31, 15, 48]
    t, q_exact, ek, ev, seq, pos = build_paged_case(rng, torch.float32, lengths, counts, heads, kv_heads, hd, page_size)
    scale = 1.0 / math.sqrt(hd)
    if broken is not None:
        at = 150        # of the first request: seen by its later tokens alone
        block, offset = t["table"][0, at // page_size].item(), at % page_size
        from microllm_rocm_amd.cache.layout import value_rows, write_value_rows
        rows = value_rows(t["v"], hd).clone()
        rows[block, :, offset, 1] = broken
        write_value_rows(t["v"], rows)
    run = lambda index, split: kernels().paged_attention_rowwise(t["q"][index].contiguous(), t["k"], t["v"], t["table"], t["seq"][index].contiguous(),
                                                                 t["pos"][index].contiguous(), scale, 0, heads, kv_heads, hd, split=split)
    together = run(slice(None), False)
    alone = torch.cat([run(slice(token, token + 1), True) for token in range(len(pos))])
    assert torch.equal(torch.nan_to_num(together, 7.0, 8.0, 9.0), torch.nan_to_num(alone, 7.0, 8.0, 9.0))
    reference = reference_attention(q_exact, ek, ev, seq, pos, heads, kv_heads, hd, scale, 0)
    sound = ~((seq == 0) & (pos >= 150)) if broken is not None else np.ones(len(pos), dtype=bool)
    np.testing.assert_allclose(together.cpu().numpy()[sound], reference[sound], rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("m,width,k,tile_rows", [(65, 24, 32, 0), (129, 200, 544, 0), (300, 129, 64, 0), (300, 512, 96, 128)])
def test_tiled_product_with_clamped_gates(m, width, k, tile_rows):
    """From the float32 sums, rounded once: half a unit of bfloat16 beside what the sums' own errors come to."""
    rng = np.random.default_rng(m)
    x_exact, x = to_bf16_exact(rng.normal(size=(m, k)))
    w_exact, w = to_bf16_exact(rng.normal(size=(2 * width, k)) * 0.3)
    got = kernels().gemm_tiled(x, kernels().pack_weight(w, interleave_halves=True), 2 * width, "clamped", tile_rows=tile_rows, limit=2.5, slope=1.7)
    product = x_exact @ w_exact.T
    gate, up = np.minimum(product[:, :width], 2.5), np.clip(product[:, width:], -2.5, 2.5)
    want = gate / (1.0 + np.exp(-1.7 * gate)) * (up + 1.0)
    assert (np.abs(got.double().cpu().numpy() - want) <= 2.0 ** -8 * np.abs(want) + 1e-4).all()
    assert float(got.float().abs().max()) > 1.0


@pytest.mark.parametrize("heads,dim,vdim", [(2, 64, 128), (3, 20, 70), (1, 16, 8), (4, 33, 129)])
@pytest.mark.parametrize("strength", [0.02, 1.0, 400.0])
def test_chunks_with_a_decay_a_channel(heads, dim, vdim, strength):
    """Requests without tokens, of one token and about a chunk's and a part's edges, each from a state of its own, against the walk
    in float64; decays close to one, of ordinary size and that leave nothing. Sums of up to 64 logarithms err by 64 roundings of
    up to 150, of which a power takes 0.7: far below the bound wherever the power is not below it itself."""
    rng = np.random.default_rng(dim)
    lengths, slots = [130, 1, 0, 64, 63, 65, 17, 200], [3, 0, 7, 5, 1, 2, 6, 8]
    cu = np.concatenate([[0], np.cumsum(lengths)])
    n, keys, values = cu[-1], heads * dim, heads * vdim
    q, k, v = (rng.normal(size=(n, heads, size)).astype(np.float32) for size in (dim, dim, vdim))
    logs = (-strength * rng.exponential(size=(n, heads, dim))).astype(np.float32)
    before = rng.normal(size=(9, heads, dim, vdim)).astype(np.float32)
    proj = device(np.concatenate([a.reshape(n, -1) for a in (q, k, v)], axis=1))
    state = device(before)
    run = lambda p, s: kernels().gla_channel_chunks(p, 0, keys, 2 * keys, device(logs.reshape(n, keys)), s, device(cu, torch.int32),
                                                    device(slots, torch.int32), len(lengths), heads, dim, vdim, 0.5)
    got = run(proj, state).cpu().numpy().reshape(n, heads, vdim)
    for index, slot in enumerate(slots):
        kept = before[slot].astype(np.float64)
        want = np.zeros((lengths[index], heads, vdim))
        for at, token in enumerate(range(cu[index], cu[index + 1])):
            kept = kept * np.exp2(logs[token].astype(np.float64))[:, :, None] + k[token][:, :, None].astype(np.float64) * v[token][:, None, :]
            want[at] = 0.5 * np.einsum("hd,hdv->hv", q[token].astype(np.float64), kept)
        assert np.abs(state[slot].cpu().numpy() - kept).max() < 2e-5 * np.abs(kept).max(), index
        if lengths[index]:
            assert np.abs(got[cu[index]:cu[index + 1]] - want).max() < 2e-5 * np.abs(want).max(), index
    assert torch.equal(state[4], device(before)[4]) and torch.equal(state[7], device(before)[7])
    # a value that is not finite reaches its own token and those after it
    for broken in (float("inf"), float("nan")):
        proj[100, 2 * keys] = broken
        after = run(proj, device(before)).cpu().numpy().reshape(n, heads, vdim)
        assert np.isfinite(after[:100]).all() and not np.isfinite(after[100, 0, 0])
        np.testing.assert_array_equal(after[130:], got[130:])
        np.testing.assert_allclose(after[:100], got[:100], rtol=0, atol=2e-5 * np.abs(got).max())


@pytest.mark.parametrize("streams", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("width", [4, 260, 1024, 2044, 2046, 6148])
@pytest.mark.parametrize("parts,rms", [(1, 0), (2, 1), (5, 0), (6, 1)])
def test_stream_norm_by_groups_of_four(streams, width, parts, rms):
    rng = np.random.default_rng(width + streams)
    x, y = rng.normal(size=(5, streams, width)).astype(np.float32), rng.normal(size=(parts, 5, width)).astype(np.float32)
    mix, give, take = rng.normal(size=(streams, streams)).astype(np.float32), rng.normal(size=streams).astype(np.float32), rng.normal(size=streams).astype(np.float32)
    weight = rng.normal(size=width).astype(np.float32)
    fresh = np.einsum("st,nsw->ntw", mix.astype(np.float64), x) + give[None, :, None].astype(np.float64) * y.astype(np.float64).sum(0)[:, None, :]

    def norm(rows):
        u = np.einsum("t,ntw->nw", take.astype(np.float64), rows)
        u = u if rms else u - u.mean(-1, keepdims=True)
        return u / np.sqrt((u ** 2).mean(-1, keepdims=True) + 1e-5) * weight

    x_device = device(x)
    got = kernels().stream_norm(x_device, device(weight), 1e-5, torch.float32, rms=bool(rms), delta=device(y), mix=device(mix), give=device(give),
                                take=device(take), write_x=True)
    np.testing.assert_allclose(x_device.cpu().numpy(), fresh, rtol=2e-5, atol=2e-5 * np.abs(fresh).max())
    np.testing.assert_allclose(got.cpu().numpy(), norm(fresh), rtol=2e-5, atol=2e-5 * np.abs(norm(fresh)).max())
    some = kernels().stream_norm(x_device, device(weight), 1e-5, torch.bfloat16, rms=bool(rms), take=device(take), rows=device([4, 0], torch.int32))
    np.testing.assert_allclose(some.float().cpu().numpy(), norm(fresh)[[4, 0]], rtol=2.0 ** -8, atol=2e-5 * np.abs(norm(fresh)).max())


@pytest.mark.parametrize("n", [1024, 16384, 16400, 20480, 36864, 36888])      # 1, 4, 5, 5, 9 and 10 tiles a workgroup, some the last one
@pytest.mark.parametrize("k", [24, 256, 264, 776])
def test_product_for_64_rows_by_tiles_a_workgroup(n, k):
    rng = np.random.default_rng(n + k)
    x_exact, x = to_bf16_exact(rng.normal(size=(64, k)))
    w_exact, w = to_bf16_exact(rng.normal(size=(n, k)))
    packed = kernels().pack_weight(w)
    plan = kernels().medium_plan(n, k, may_split=False)
    whole = kernels().gemm_medium(x, packed, n, "f32", plan=plan)
    bound = (k + 1) * F32_STEP * (np.abs(x_exact) @ np.abs(w_exact).T)
    assert (np.abs(whole.double().cpu().numpy() - x_exact @ w_exact.T) <= bound).all()
    for m in (16, 17, 33, 48):
        assert torch.equal(kernels().gemm_medium(x[:m].contiguous(), packed, n, "f32", plan=plan), whole[:m]), m


@pytest.mark.parametrize("rank", [1, 4, 15, 16, 17, 20, 32, 37])
@pytest.mark.parametrize("n_tokens", [1, 7, 8, 9, 600, 33001])       # the last: several tokens a thread from rank 4 on
def test_decays_of_every_rank_and_of_infinite_inputs(rank, n_tokens):
    """Whole and broken groups of 16 numbers of the low rank, whole and broken groups of tokens. An input that is infinite drives
    a channel's decay to zero or one by its weight's sign; one that is no number leaves none."""
    rng = np.random.default_rng(rank)
    channels, tau, offset = 130, 16.0, 3
    low, a2, bias = rng.normal(size=(n_tokens, rank)), rng.normal(size=(channels, rank)), rng.normal(size=channels)
    low[n_tokens - 1, rank - 1] = np.inf
    low[n_tokens // 2, 0] = -np.inf
    proj = np.concatenate([rng.normal(size=(n_tokens, offset)), low], axis=1).astype(np.float32)
    low, a2, bias = (value.astype(np.float32).astype(np.float64) for value in (low, a2, bias))
    with np.errstate(over="ignore", invalid="ignore"):      # infinity less infinity, where one token and one number have both
        z = low @ a2.T + bias
        logs = -np.logaddexp(0.0, -z) / tau
    for base_two, want in ((False, np.exp(logs)), (True, logs / math.log(2.0))):
        got = kernels().gla_decay(device(proj), offset, device(a2), device(bias), tau, base_two=base_two).double().cpu().numpy()
        # rank + 2 roundings of z's terms and a few of the logarithm's and the power's own
        bound = (rank + 8) * 2 * F32_STEP * (np.abs(np.nan_to_num(low, posinf=0, neginf=0)) @ np.abs(a2).T + np.abs(bias) + 1.0)
        finite = np.isfinite(want)
        assert (np.abs(got[finite] - want[finite]) <= bound[finite]).all()
        np.testing.assert_array_equal(np.where(finite, 0.0, got), np.where(finite, 0.0, want))


@pytest.mark.parametrize("strong_first", [1, 3, 4, 12, 15])
@pytest.mark.parametrize("strong", [20.0, 150.0, 4000.0])
def test_chunks_where_slow_decays_follow_strong_ones(strong_first, strong):
    """Every 16 tokens begin with some that leave (next to) nothing, then decays close to one. A weight between two tokens errs by the
    roundings of the logarithms between them alone, however strong those before: 2^-24 for each of up to 64 sums of an exponent x,
    times x log 2 relative to the term; products, powers and the sums over channels and tokens add at most 48 roundings."""
    rng = np.random.default_rng(strong_first)
    heads, dim, vdim, n = 2, 4, 8, 64
    keys, values = heads * dim, heads * vdim
    q, k, v = (rng.normal(size=(n, heads, size)).astype(np.float32) for size in (dim, dim, vdim))
    logs = (-0.01 * rng.exponential(size=(n, heads, dim))).astype(np.float32)
    strong_ones = np.arange(n) % 16 < strong_first
    logs[strong_ones] = -strong * rng.uniform(0.9, 1.0, size=(strong_ones.sum(), heads, dim))
    proj = device(np.concatenate([a.reshape(n, -1) for a in (q, k, v)], axis=1))
    state = torch.zeros((1, heads, dim, vdim), device=DEVICE)
    got = kernels().gla_channel_chunks(proj, 0, keys, 2 * keys, device(logs.reshape(n, keys)), state, device([0, n], torch.int32), device([0], torch.int32), 1,
                                       heads, dim, vdim, 1.0).double().cpu().numpy().reshape(n, heads, vdim)
    q, k, v, logs = (a.astype(np.float64) for a in (q, k, v, logs))
    before = np.concatenate([np.zeros((1, heads, dim)), np.cumsum(logs, axis=0)])
    exponents = before[1:, None] - before[None, 1:]                       # [t, j, head, channel]: the logarithms of tokens j + 1 .. t
    pairs = np.where(np.tri(n, dtype=bool)[:, :, None, None], np.exp2(np.minimum(exponents, 0.0)), 0.0)
    roundings = 48 + 64 * math.log(2.0) * np.abs(exponents)
    want = np.einsum("thd,jhd,tjhd,jhv->thv", q, k, pairs, v)
    bound = np.einsum("thd,jhd,tjhd,jhv->thv", np.abs(q), np.abs(k), pairs * roundings, np.abs(v)) * F32_STEP
    assert (np.abs(got - want) <= bound).all(), float((np.abs(got - want) / bound).max())
    left = np.einsum("jhd,jhd,jhv->hdv", k, pairs[-1], v)
    bound = np.einsum("jhd,jhd,jhv->hdv", np.abs(k), (pairs * roundings)[-1], np.abs(v)) * F32_STEP
    assert (np.abs(state[0].double().cpu().numpy() - left) <= bound).all()


@pytest.mark.parametrize("tiles", [127, 128, 129, 256, 257, 384, 385, 512, 513, 768, 769])       # half tiles up to 128, two a workgroup from 257 to 512 and from 769
@pytest.mark.parametrize("m", [1, 5, 6, 9, 16])
def test_streaming_epilogues_by_tiles(tiles, m):
    """The residual and the q/k/v epilogue on both sides of the lines where a workgroup takes half a tile, one and two, against
    the plain product (the same sums to the bit) and the kernels that they replace."""
    rng = np.random.default_rng(tiles + m)
    ka, n, k = kernels(), 16 * tiles, 1536
    _, x = to_bf16_exact(rng.normal(size=(m, k)))
    _, w = to_bf16_exact(rng.normal(size=(n, k)) * 0.1)
    packed = ka.pack_weight(w)
    product = ka.gemm_skinny(x, packed, n, "f32")
    stream, norm = rng.normal(size=(m, n)), device(rng.normal(size=n))
    if n <= 8192:
        h = device(stream)
        values, scale = ka.gemm_skinny_residual(x, packed, h, norm, n, 1e-5)
        assert torch.equal(h, device(stream) + product)
        assert torch.equal(values, (h * norm).to(torch.bfloat16))
        # the sums of squares, through a product that applies the rows' factors to the identity's columns
        eye = ka.pack_weight(torch.eye(n, dtype=torch.bfloat16, device=DEVICE)[:16].contiguous())
        factor = 1.0 / torch.sqrt(h.double().pow(2).mean(1, keepdim=True) + 1e-5)
        got = ka.gemm_skinny(values, eye, 16, "f32", scale=scale).double()
        assert torch.allclose(got, values[:, :16].double() * factor, rtol=(n / 8 + 8) * 2 * F32_STEP, atol=0.0)
    heads, hd, rotary = tiles, 16, 16
    order = ka.rotary_pair_order(heads, 0, hd, rotary // 2)
    positions = device(rng.integers(0, 30000, size=m), torch.int32)
    table = ka.rope_table(positions, device(1e4 ** -(np.arange(0, rotary, 2) / rotary), torch.float64))
    bias = device(rng.normal(size=n))
    one = ka.gemm_skinny_qkv(x, ka.pack_weight(w, row_order=order), bias, None, table, None, None, heads, 0, hd, 16)
    two = ka.qkv_rope_store(product, bias, positions, None, device(1e4 ** -(np.arange(0, rotary, 2) / rotary), torch.float64), None, None, heads, 0, hd, 16,
                            torch.bfloat16)
    assert torch.equal(one, two)


def whole_numbers(generator, *shape):
    """-1, 0 and 1 in bfloat16: products whose float32 sums are exact whatever their order."""
    return torch.randint(-1, 2, shape, generator=generator, device=DEVICE).to(torch.bfloat16)


@pytest.mark.parametrize("n", [40, 2064])        # half and whole tiles
def test_streaming_product_of_the_longest_reductions(n):
    """Byte offsets of 2^30 and more, where the kernel's 32-bit offsets end: the same sums with 64-bit addresses."""
    generator = torch.Generator(device=DEVICE).manual_seed(n)
    k = (1 << 23) + 40 if n == 40 else (1 << 23) + 8
    x = whole_numbers(generator, 20, k)
    w = torch.zeros((n, k), dtype=torch.bfloat16, device=DEVICE)
    w[:40] = whole_numbers(generator, 40, k)
    w[n - 1, k - 3:] = 1.0
    packed = kernels().pack_weight(w)
    want = torch.cat([x.float() @ part.float().T for part in w.split(64)], dim=1)
    del w
    for m in (1, 9, 20):
        assert torch.equal(kernels().gemm_skinny(x[:m].contiguous(), packed, n, "f32"), want[:m])
        assert torch.equal(kernels().gemm_skinny(x[:m].contiguous(), packed, n, "bf16"), want[:m].to(torch.bfloat16))


# Tiles of a workgroup, unsplit and in three parts: up to four, workgroups of four waves; up to eight, of eight; more, of eight with two tiles each.
@pytest.mark.parametrize("n,tiles,of_parts", [(40, 1, 1), (16 * 300, 2, 4), (16 * 700 - 8, 3, 9), (16 * 1500 - 8, 6, 12), (16 * 2100, 9, 9)])
@pytest.mark.parametrize("k", [8, 256, 264, 512, 520, 768, 1000, 1280])       # one to five stages of 256, whole and begun
def test_product_for_64_rows_of_any_number_of_stages(n, tiles, of_parts, k):
    """Two stages a round and what is left of an odd number; sums of whole numbers, which have no rounding to differ in."""
    chosen = library.load().mll_gemm_medium_tiles
    assert all(chosen(m, n, k, 2, 8, 1) == tiles for m in (17, 32, 33, 64)) and chosen(64, n, 1000, 2, 8, 3) == of_parts
    generator = torch.Generator(device=DEVICE).manual_seed(n + k)
    x, w = whole_numbers(generator, 64, k), whole_numbers(generator, n, k)
    packed, want = kernels().pack_weight(w), x.float() @ w.float().T
    for m in (17, 32, 33, 64):
        for splits in (1, 2, 3):
            got = kernels().gemm_medium(x[:m].contiguous(), packed, n, "f32", plan=(2, 8, splits))
            assert torch.equal(got.sum(0) if splits > 1 else got, want[:m])


@pytest.mark.parametrize("n,splits", [(40, 1), (40, 16), (200, 2)])
def test_product_for_64_rows_of_the_longest_reductions(n, splits):
    """Where a workgroup's tiles pass what 32-bit offsets reach: the same sums with 64-bit addresses, whole and in parts."""
    generator = torch.Generator(device=DEVICE).manual_seed(n)
    k = (1 << 21) + 40
    x, w = whole_numbers(generator, 64, k), whole_numbers(generator, n, k)
    packed = kernels().pack_weight(w)
    want = x.float() @ w.float().T
    for m in (17, 64):
        got = kernels().gemm_medium(x[:m].contiguous(), packed, n, "f32", plan=(2, 8, splits))
        assert torch.equal(got.sum(0) if splits > 1 else got, want[:m])
    if splits == 1:
        assert torch.equal(kernels().gemm_medium(x, packed, n, "bf16"), want.to(torch.bfloat16))


@pytest.mark.parametrize("rows,n,k", [(512, 19456, 896), (1024, 8192, 2048)])
def test_gated_products_of_rows_at_any_address(rows, n, k):
    """Rows that begin at no 16-byte boundary go to the library, whose product rounds gate and up first: a unit of bfloat16 each, and
    the sums' own errors, beside the tiled kernel's result for the same rows at a boundary."""
    from microllm_rocm_amd.parts.linear import Weight, linear, linear_clamped_glu, takes_tiled
    rng = np.random.default_rng(rows)
    _, x = to_bf16_exact(rng.normal(size=(rows, k)))
    _, w = to_bf16_exact(rng.normal(size=(n, k)) * k ** -0.5)
    weight = Weight(w, gated=True)
    apart = torch.empty(rows * k + 1, dtype=torch.bfloat16, device=DEVICE)[1:].view(rows, k)
    apart.copy_(x)
    assert takes_tiled(x, weight) and takes_tiled(x, weight, from_float=True) and apart.data_ptr() % 16 != 0
    for product in (lambda rows_: linear(rows_, weight, gated=True), lambda rows_: linear_clamped_glu(rows_, weight, 7.0, 1.7)):
        got, want = product(apart).float(), product(x).float()
        assert bool(((got - want).abs() <= 2.0 ** -6 * want.abs() + 2.0 ** -6 * 0.1).all())


@pytest.mark.parametrize("rows", [49, 64])
@pytest.mark.parametrize("n,k", [(4096, 128), (8192, 1000)])      # 256 tiles, from which the packed copy takes 49 rows and more
def test_gated_products_of_49_to_64_rows_at_any_address(rows, n, k):
    """Rows that begin at no 16-byte boundary go to the library, which rounds gate g and up first: two roundings of 2^-9 beside the
    results' own two, of which |g silu'(g)| <= 1.3 |silu(g)| + 0.3 makes less than the bound for every |up| below 5."""
    from microllm_rocm_amd.parts.linear import Weight, linear, takes_packed
    rng = np.random.default_rng(rows)
    _, x = to_bf16_exact(rng.normal(size=(rows, k)))
    _, w = to_bf16_exact(rng.normal(size=(n, k)) * k ** -0.5)
    weight = Weight(w, gated=True)
    apart = torch.empty(rows * k + 1, dtype=torch.bfloat16, device=DEVICE)[1:].view(rows, k)
    apart.copy_(x)
    assert takes_packed(weight, rows, True, x.data_ptr()) and not takes_packed(weight, rows, True, apart.data_ptr())
    got, want = linear(apart, weight, gated=True).float(), linear(x, weight, gated=True).float()
    assert bool(((got - want).abs() <= 2.0 ** -6 * want.abs() + 2.0 ** -6 * 0.1).all())

# ---- decode attention: both sides of the line past which pages are read past the caches, with and without a bias ----
@pytest.mark.parametrize("heads,kv_heads,hd,page_size,splits,biased", [
    (4, 4, 64, 16, 8, False), (4, 4, 64, 16, 3, True), (8, 4, 128, 32, 5, True), (8, 4, 128, 16, 4, False), (8, 4, 128, 16, 8, True), (8, 4, 128, 32, 9, False), (2, 2, 192, 48, 19, True),
    (3, 3, 48, 16, 11, True), (5, 1, 256, 16, 16, False), (18, 1, 80, 16, 9, True)])
def test_decode_attention_reads_every_line_of_its_pages(heads, kv_heads, hd, page_size, splits, biased):
    rng = np.random.default_rng(heads + hd + splits)
    lengths = [417, 1, 33, 260, 16, 31, 129, 8]
    t, q_exact, ek, ev, seq, pos = build_paged_case(rng, torch.bfloat16, lengths, [1] * len(lengths), heads, kv_heads, hd, page_size)
    scale, longest = 1.0 / math.sqrt(hd), 90
    table = rng.normal(size=(longest + 1, heads)).astype(np.float32) if biased else np.zeros((longest + 1, heads), np.float32)
    want = np.zeros((len(lengths), heads, hd))
    for token, length in enumerate(lengths):
        distance = np.minimum(length - 1 - np.arange(length), longest)
        for head in range(heads):
            scores = ek[token][:, head // (heads // kv_heads)] @ q_exact[token].reshape(heads, hd)[head] * scale + table[distance, head]
            weights = np.exp(scores - scores.max())
            want[token, head] = weights / weights.sum() @ ev[token][:, head // (heads // kv_heads)]
    k = kernels()
    extras = k.AttentionExtras(bias=torch.tensor(table, device=DEVICE)) if biased else None
    out = torch.zeros_like(t["q"])
    k.paged_attention_decode(t["q"], t["k"], t["v"], t["table"], t["seq"], t["pos"], scale, 0, heads, kv_heads, hd, splits, out=out, extras=extras)
    np.testing.assert_allclose(out.float().cpu().numpy(), want.reshape(len(lengths), -1), **tolerance(torch.bfloat16))



@pytest.mark.parametrize("heads,kv_heads,hd,page_size,window,splits", [
    (28, 4, 128, 16, 0, 1), (14, 2, 64, 16, 0, 1), (14, 2, 64, 48, 0, 2), (8, 4, 128, 32, 260, 1), (16, 4, 256, 16, 0, 1), (5, 5, 48, 16, 0, 1)])
def test_decode_attention_of_waves_with_any_number_of_pairs(heads, kv_heads, hd, page_size, window, splits):
    """A workgroup's four waves take pairs of tiles of 16 keys in turn, two a round and what is left of an odd number: none to five a wave, alike and one
    more for some of the waves, the last pair's keys one or all."""
    rng = np.random.default_rng(heads + hd + window)
    lengths = [1, 32, 33, 128, 129, 160, 256, 257, 289, 384, 385, 512, 513, 609]
    t, q_exact, ek, ev, seq, pos = build_paged_case(rng, torch.bfloat16, lengths, [1] * len(lengths), heads, kv_heads, hd, page_size)
    out = kernels().paged_attention_decode(t["q"], t["k"], t["v"], t["table"], t["seq"], t["pos"], hd ** -0.5, window, heads, kv_heads, hd, splits)
    want = reference_attention(q_exact, ek, ev, seq, pos, heads, kv_heads, hd, hd ** -0.5, window)
    np.testing.assert_allclose(out.float().cpu().numpy(), want, **tolerance(torch.bfloat16))


@pytest.mark.parametrize("heads,kv_heads,hd,tokens,splits", [(28, 4, 128, 4, 8), (14, 2, 64, 12, 8)])
def test_decode_attention_of_long_steps_has_the_bits_of_fewer_tokens(heads, kv_heads, hd, tokens, splits):
    """128 and 192 workgroups of a step planned for 8192 positions, from which pages are read past the caches, and one token less."""
    rng, k = np.random.default_rng(hd), kernels()
    t, *_ = build_paged_case(rng, torch.bfloat16, [8100] + [70] * (tokens - 1), [1] * tokens, heads, kv_heads, hd, 16)
    table = torch.full((tokens, 512), -1, dtype=torch.int32, device=DEVICE)
    table[:, :t["table"].shape[1]] = t["table"]
    run = lambda n: k.paged_attention_decode(t["q"][:n], t["k"], t["v"], table, t["seq"][:n], t["pos"][:n], hd ** -0.5, 0, heads, kv_heads, hd, splits)
    assert torch.equal(run(tokens)[:tokens - 1], run(tokens - 1))


# ---- experts in large tiles, of 128 rows and one a workgroup: remainders, experts without a pair, ids that return their input ----
@pytest.mark.parametrize("n,width,ff,experts,top,identity,gated", [
    (700, 128, 384, 3, 2, 0, True), (520, 256, 128, 2, 1, 1, True), (1300, 128, 264, 5, 2, 2, False),
    (129, 384, 128, 1, 1, 0, True), (3000, 128, 256, 4, 2, 1, True)])
def test_experts_in_large_tiles(n, width, ff, experts, top, identity, gated):
    """Against the kernels that take a pair at a time, whose sums have another order; and the bits of the same pairs in steps too small for
    the large tiles, which the smaller ones take."""
    k, rng = kernels(), np.random.default_rng(n + ff)
    x = device(rng.normal(size=(n, width)), torch.bfloat16)
    gate_up = device(rng.normal(size=(experts, (2 if gated else 1) * ff, width)) * 0.2, torch.bfloat16)
    down = device(rng.normal(size=(experts, width, ff)) * 0.2, torch.bfloat16)
    ids = np.argsort(rng.random((n, experts + identity)) + np.linspace(0, 0.9, experts + identity), axis=1)[:, :top]      # the last ones are rarely chosen
    ids = device(np.where((ids == experts - 1) & (experts > 3), 0, ids), torch.int32)       # and one never
    weights = device(rng.uniform(0.2, 1.5, size=(n, top)))
    for on_input in (False, True):
        options = dict(gated=gated, activation="silu", identity=identity)
        if on_input and identity:
            continue
        tiled = k.moe_experts(x, ids, weights, gate_up, down, on_input, grouped=True, **options)
        one_by_one = k.moe_experts(x, ids, weights, gate_up, down, on_input, grouped=False, **options)
        assert float((tiled - one_by_one).abs().max()) < 0.02 * float(one_by_one.abs().max())      # the inner values are rounded from sums in another order
        few = 100 * experts // top       # below 128 pairs an expert
        small = k.moe_experts(x[:few], ids[:few].contiguous(), weights[:few].contiguous(), gate_up, down, on_input, grouped=True, **options)
        assert few < n and torch.equal(small, tiled[:, :few])


def tiling(counts, n_out, columns):
    """The height that the kernel chooses for experts of ``counts`` pairs, and how many tiles that makes: the first of those whose rounds of 256
    workgroups cost least, a round as much as a stage of its rows and of 256 of the weight."""
    blocks, best = -(-n_out // columns), None
    for height in (256, 192, 128):
        tiles = sum(-(-count // height) for count in counts) * blocks
        cost = -(-tiles // 256) * (height + 256)
        if best is None or cost < best[0]:
            best = (cost, height, tiles)
    return best[1:]


ENDS_OF_256 = [600, 577, 640, 641, 700, 704, 705, 768, 0, 767, 1, 650, 740, 600, 768, 690]      # last tiles of up to 128, 192 and 256 rows, and of one
ENDS_OF_192 = [192, 129, 191, 0, 190, 128, 192, 1, 180, 192] * 3
ENDS_OF_128 = [128] * 29 + [129]
MANY_EXPERTS = [(140 * e) % 331 if e % 9 else 0 for e in range(70)]          # experts on both sides of a wave's lanes, some without a pair


# which product has more tiles than there are workgroups, and their height: gate and up (or up alone), or down
@pytest.mark.parametrize("counts,width,ff,gated,identity,walks,height", [
    (ENDS_OF_256, 128, 2048, True, 0, "inner", 256), (ENDS_OF_256, 4096, 128, True, 37, "down", 256), (ENDS_OF_256, 128, 4096, False, 0, "inner", 256),
    (ENDS_OF_192, 128, 2048, True, 0, "inner", 192), (ENDS_OF_192, 4096, 128, True, 0, "down", 192),
    (ENDS_OF_128, 128, 2048, True, 0, "inner", 128), (ENDS_OF_128, 4096, 128, False, 5, "down", 128), (MANY_EXPERTS, 128, 896, True, 40, "inner", 192)])
def test_experts_in_more_large_tiles_than_workgroups(counts, width, ff, gated, identity, walks, height):
    """A workgroup goes from tile to tile, whose rows and results take the LDS of the tile before: against the kernels that take a pair at a time, and the
    bits of fewer pairs, which smaller tiles take."""
    k, experts = kernels(), len(counts)
    inner, outer = tiling(counts, ff, 128 if gated else 256), tiling(counts, width, 256)
    chosen, tiles = inner if walks == "inner" else outer
    assert chosen == height and tiles > 256 and sum(counts) + identity >= 128 * experts
    generator = torch.Generator(device=DEVICE).manual_seed(width + ff + experts)
    normal = lambda *shape: torch.randn(shape, generator=generator, device=DEVICE)
    ids = torch.cat([torch.full((count,), e, dtype=torch.int32) for e, count in enumerate([*counts, identity])]).to(DEVICE)
    ids = ids[torch.randperm(len(ids), generator=generator, device=DEVICE)][:, None].contiguous()
    n = ids.shape[0]
    x, weights = normal(n, width).to(torch.bfloat16), normal(n, 1).abs() + 0.2
    gate_up, down = ((normal(experts, rows, terms) * terms ** -0.5).to(torch.bfloat16) for rows, terms in (((2 if gated else 1) * ff, width), (width, ff)))
    for on_input in (False, True) if identity == 0 else (False,):
        run = lambda rows, grouped: k.moe_experts(x[:rows], ids[:rows], weights[:rows], gate_up, down, on_input, grouped=grouped, gated=gated, activation="silu",
                                                  identity=1 if identity else 0)
        tiled, one_by_one = run(n, True), run(n, False)
        assert float((tiled - one_by_one).abs().max()) < 0.02 * float(one_by_one.abs().max())      # the inner values are rounded from sums in another order
        few = 128 * experts - 1
        assert few < n and experts * -(-max((2 if gated else 1) * ff, width) // 256) < 512        # the smaller tiles take so few
        assert torch.equal(run(few, True), tiled[:, :few])


def test_queries_keys_and_values_of_more_tiles_than_workgroups():
    """The tiled product's epilogue with rotation and pages where a workgroup takes a second tile (17 x 18 of 128 rows), against tiles of 256 (9 x 18), which fit one
    round, and against the two kernels it replaces."""
    k, generator = kernels(), torch.Generator(device=DEVICE).manual_seed(5)
    heads, kv_heads, hd, hidden, m, page = 28, 4, 128, 64, 2100, 16
    total = (heads + 2 * kv_heads) * hd
    normal = lambda *shape: torch.randn(shape, generator=generator, device=DEVICE)
    x, bias = normal(m, hidden).to(torch.bfloat16), normal(total)
    packed = k.pack_weight((normal(total, hidden) * 0.2).to(torch.bfloat16), row_order=k.rotary_pair_order(heads, kv_heads, hd, hd // 2))
    table = k.rope_table(torch.arange(m, dtype=torch.int32, device=DEVICE), 1e4 ** -(torch.arange(0, hd, 2, device=DEVICE, dtype=torch.float64) / hd))
    slots = torch.randperm(m, generator=generator, device=DEVICE).to(torch.int32)
    pages = lambda: [torch.full(shape(-(-m // page), kv_heads, page, hd), 7.0, dtype=torch.bfloat16, device=DEVICE) for shape in (key_page_shape, value_page_shape)]
    results = []
    for rows in (128, 256):
        kept = pages()
        results.append([k.gemm_tiled_qkv(x, packed, bias, slots, table, *kept, heads, kv_heads, hd, page, tile_rows=rows), *kept])
    kept = pages()
    results.append([k.qkv_rope_store(k.gemm_tiled(x, packed, total, "f32"), bias, torch.arange(m, dtype=torch.int32, device=DEVICE), slots, None, *kept, heads, kv_heads,
                                     hd, page, torch.bfloat16, pair_order=True, cos_sin=table), *kept])
    for other in results[1:]:
        assert all(torch.equal(a, b) for a, b in zip(results[0], other))


@pytest.mark.parametrize("k", [32, 64, 96, 128, 160, 192, 256, 352])
@pytest.mark.parametrize("m,n", [(2200, 8192), (2048, 8448), (2100, 8210)])
def test_tiles_whose_loads_go_out_before_the_tile_before_is_stored(m, n, k):
    """One to six stages, odd numbers of k steps, whole tiles and ragged ones, of which workgroups take a second or third: the bits of the same rows and columns
    by fewer tiles than workgroups, which each take one."""
    ka, generator = kernels(), torch.Generator(device=DEVICE).manual_seed(m + n + k)
    x, w = ((torch.randn(shape, generator=generator, device=DEVICE) * scale).to(torch.bfloat16) for shape, scale in (((m, k), 1.0), ((n, k), k ** -0.5)))
    packed, band = ka.pack_weight(w), 512
    for epilogue, tile_rows in (("gated", 256), ("gated", 128), ("bf16", 256), ("f32", 160)):
        whole = ka.gemm_tiled(x, packed, n, epilogue, tile_rows=tile_rows)
        width = band // 2 if epilogue == "gated" else band
        for rows in (slice(0, 300), slice(m - 300, m)):
            for at in (0, n // 2 // band * band, (n - 1) // band * band):
                part = ka.gemm_tiled(x[rows].contiguous(), packed[at // 16:(at + band) // 16].contiguous(), min(band, n - at), epilogue, tile_rows=tile_rows)
                assert torch.equal(part, whole[rows, at * width // band:at * width // band + part.shape[1]]), (epilogue, rows, at)
    assert float((ka.gemm_tiled(x, packed, n, "f32") - x.float() @ w.float().T).abs().max()) < 1e-5 * k ** 0.5 + 1e-4      # sums of at most 352 products of size 1 / sqrt(k)


@pytest.mark.parametrize("k", [32, 64, 96, 160, 352])
@pytest.mark.parametrize("tile_rows", [128, 160, 256])
def test_infinities_at_the_end_of_a_reduction_stay_infinities(k, tile_rows):
    """A stage takes two steps of 32: one that has only one multiplies nothing by the zeros of the other. One infinity in a row is that of its sign and the
    weight's in every column, other rows keep their bits."""
    ka, generator = kernels(), torch.Generator(device=DEVICE).manual_seed(k)
    m, n = 300, 520
    x, w = (torch.randn(shape, generator=generator, device=DEVICE).to(torch.bfloat16) for shape in ((m, k), (n, k)))
    w = torch.where(w == 0, torch.ones_like(w), w)
    packed, spoilt = ka.pack_weight(w), x.clone()
    places = {row: place for row, place in ((1, k - 1), (2, k - 32), (130, k - 33), (4, k - 64), (5, 0), (m - 1, k - 1)) if place >= 0}
    for row, place in places.items():
        spoilt[row, place] = math.inf if row % 2 else -math.inf
    kept = torch.tensor([row for row in range(m) if row not in places], device=DEVICE)
    for epilogue, splits in (("f32", 1), ("bf16", 1), ("f32", 2)):
        options = dict(epilogue=epilogue, splits=splits, tile_rows=tile_rows)
        whole, got = (ka.gemm_tiled(rows, packed, n, **options) for rows in (x, spoilt))
        assert torch.equal(got[..., kept, :], whole[..., kept, :])
        total = got.sum(0) if splits > 1 else got.float()
        for row, place in places.items():
            assert torch.equal(total[row], w[:, place].float().sign() * float(spoilt[row, place])), (epilogue, splits, row)


@pytest.mark.parametrize("heads,kv_heads,hd,window", [(14, 2, 64, 0), (4, 2, 48, 100), (4, 1, 128, 0), (2, 1, 256, 33)])
def test_prompts_in_tiles_of_half_the_queries_have_the_same_bits(heads, kv_heads, hd, window):
    """Tiles of 64 queries, whose second one in a workgroup goes to the waves from the last on, against tiles of 128."""
    rng, k = np.random.default_rng(hd + window), kernels()
    lengths, counts = [517, 300, 97, 64, 131, 33], [130, 300, 65, 64, 128, 1]
    t, *_ = build_paged_case(rng, torch.bfloat16, lengths, counts, heads, kv_heads, hd, 16)
    results = []
    for rows in (128, 64):
        tiles, start = [], 0
        for index, (length, count) in enumerate(zip(lengths, counts)):
            tiles += [(index, start + offset, min(rows, count - offset), length - count + offset) for offset in range(0, count, rows)]
            start += count
        pairs = torch.tensor(k.pair_query_tiles(tiles, adjacent=window > 0), dtype=torch.int32, device=DEVICE)
        results.append(k.paged_attention_prefill(t["q"], t["k"], t["v"], t["table"], pairs, t["pos"], hd ** -0.5, window, heads, kv_heads, hd))
    assert torch.equal(*results)


@pytest.mark.parametrize("heads,kv_heads,hd", [(28, 4, 16), (33, 3, 32), (28, 4, 48)])
def test_prompts_have_the_same_bits_in_steps_of_few_and_of_many_workgroups(heads, kv_heads, hd):
    """Heads of up to 32 are worked on without whole blocks from 257 workgroups on: all of a step's entries in one launch, and by few."""
    k, lengths = kernels(), [1300, 517, 129, 1100]
    t, *_ = build_paged_case(np.random.default_rng(hd), torch.bfloat16, lengths, lengths, heads, kv_heads, hd, 16)
    tiles = torch.tensor(k.pair_query_tiles(query_tile_list(lengths, lengths)), dtype=torch.int32, device=DEVICE)
    few = 256 // heads
    assert len(tiles) * heads > 256
    run = lambda some, out: k.paged_attention_prefill(t["q"], t["k"], t["v"], t["table"], some, t["pos"], hd ** -0.5, 0, heads, kv_heads, hd, out=out)
    parts = torch.empty_like(t["q"])
    for first in range(0, len(tiles), few):
        run(tiles[first:first + few].contiguous(), parts)
    assert torch.equal(run(tiles, torch.empty_like(t["q"])), parts)


@pytest.mark.parametrize("heads,kv_heads", [(28, 4), (14, 2), (16, 4), (64, 8), (9, 1), (16, 16), (48, 24), (12, 6), (15, 5), (7, 7)])
def test_prefill_workgroups_take_the_longest_entries_of_all_heads_first(heads, kv_heads):
    """Every entry and head once, whatever their numbers; of a round over the eight dies none takes an earlier entry than the round before; and where the kv
    heads divide among the dies, a die keeps to its own."""
    order = library.load().mll_paged_attention_prefill_order
    for entries in (1, 2, 3, 7, 17, 33, 34):
        taken, number = [], 0
        while (item := order(entries, heads, kv_heads, ctypes.c_int64(number))) >= 0:
            taken.append(item)
            number += 1
        assert sorted(taken) == list(range(entries * heads)) + [len(taken)] * (len(taken) - entries * heads)
        rounds = [[item // heads for item in taken[i:i + 8] if item < entries * heads] for i in range(0, len(taken), 8)]
        assert all(max(now) <= min(after) for now, after in zip(rounds, rounds[1:]) if now and after)
        if 8 % kv_heads == 0 or kv_heads % 8 == 0:
            own = [{item % heads // (heads // kv_heads) for item in taken[die::8] if item < entries * heads} for die in range(8)]
            assert all(len(kv) <= max(1, kv_heads // 8) for kv in own)


@pytest.mark.parametrize("heads,kv_heads,hd,page_size", [(4, 2, 16, 16), (3, 1, 48, 48), (14, 2, 64, 32), (6, 3, 96, 16), (7, 7, 112, 64), (28, 4, 128, 16)])
@pytest.mark.parametrize("window", [0, 333])
def test_blocks_seen_whole_have_the_bits_of_their_runs(heads, kv_heads, hd, page_size, window):
    """Blocks of 128 keys that a wave sees whole are worked on as one, overlapped; with extras (here a bias of nothing) every run of keys by itself. Portions begin
    and end within blocks; the larger scores move their maxima by more."""
    k = kernels()
    lengths, counts = [700, 517, 131, 129, 258], [700, 130, 2, 129, 97]
    for larger in (1.0, 16.0):
        t, *_ = build_paged_case(np.random.default_rng(hd + window), torch.bfloat16, lengths, counts, heads, kv_heads, hd, page_size)
        t["q"].mul_(larger)
        tiles = torch.tensor(k.pair_query_tiles(query_tile_list(lengths, counts), adjacent=window > 0), dtype=torch.int32, device=DEVICE)
        run = lambda **more: k.paged_attention_prefill(t["q"], t["k"], t["v"], t["table"], tiles, t["pos"], hd ** -0.5, window, heads, kv_heads, hd, **more)
        nothing = k.AttentionExtras(bias=torch.zeros(2, heads, device=DEVICE))
        assert torch.equal(run(), run(extras=nothing, out=torch.empty_like(t["q"]))), larger


@pytest.mark.parametrize("heads,hd,bias", [(64, 128, False), (64, 128, True), (65, 144, False), (80, 112, False)])
def test_prompts_in_pages_beyond_32_bits(heads, hd, bias):
    """Pages of more than 2^31 elements, so that a page and its last heads begin beyond what 32 bits count in elements, and in bytes: the bits of pages of 16."""
    k, length, large = kernels(), 300, 1 << 18
    assert heads * large * hd >= 1 << 31
    t, *_ = build_paged_case(np.random.default_rng(hd), torch.bfloat16, [length], [length], heads, heads, hd, 16, spare_pages=0)
    tiles = torch.tensor(k.pair_query_tiles(query_tile_list([length], [length])), dtype=torch.int32, device=DEVICE)
    extras = k.AttentionExtras(bias=torch.linspace(-1, 1, 50 * heads, device=DEVICE).view(50, heads)) if bias else None
    run = lambda key, value, table: k.paged_attention_prefill(t["q"], key, value, table, tiles, t["pos"], hd ** -0.5, 0, heads, heads, hd, extras=extras,
                                                              out=torch.empty_like(t["q"]))
    want, order, last = run(t["k"], t["v"], t["table"]), t["table"][0, :-(-length // 16)].long(), 1
    pools = []
    for shape, small in ((key_page_shape, t["k"]), (value_page_shape, t["v"])):
        pools.append(torch.empty(shape(last + 1, heads, large, hd), dtype=torch.bfloat16, device=DEVICE))
        pools[-1][last, :, :len(order)] = small[order, :, 0].transpose(0, 1)
    try:
        assert torch.equal(run(*pools, torch.tensor([[last]], dtype=torch.int32, device=DEVICE)), want)
    finally:
        del pools
        torch.cuda.empty_cache()


@pytest.mark.parametrize("heads,kv_heads,dim,page,options", [
    (16, 4, 128, 16, dict(weights=True, temperature=True)), (9, 3, 96, 48, dict(bias=True, rot=64)), (5, 1, 16, 32, dict(values_normed=True, rot=16)),
    (7, 7, 256, 16, dict(norm_turned=True, rot=128)), (13, 2, 72, 16, dict(queries_only=True)), (8, 2, 112, 64, dict(norm_turned=True, rot=112, weights=True))])
def test_heads_of_eight_tokens_a_wave_have_the_bits_of_a_wave_each(heads, kv_heads, dim, page, options):
    """A step of many rows, of whose heads a wave takes eight tokens, against the same rows by few, whose heads have a wave each: requests that begin and end within
    eight places, pages in any order, rows without a place, places that are not one after the other."""
    k, generator = kernels(), torch.Generator(device=DEVICE).manual_seed(dim + heads)
    alone, rot = options.get("queries_only", False), options.get("rot", 0)
    n, vectors = 9000 if heads < 8 and kv_heads == 1 else 4200, heads + (0 if alone else 2 * kv_heads)
    assert -(-n // 8) * vectors >= 4096 > -(-125 // 8) * vectors        # both sides of the line
    normal = lambda *shape: torch.randn(shape, generator=generator, device=DEVICE)
    pages = -(-n // page) + 8
    rows, positions = normal(n, vectors * dim), torch.arange(n, dtype=torch.int32, device=DEVICE) * 3
    order = torch.randperm(pages, generator=generator, device=DEVICE)
    slots = (order[:, None] * page + torch.arange(page, device=DEVICE)).view(-1).to(torch.int32)
    slots = torch.cat([slots[5:1003], slots[1008:1017], slots[1030:]])[:n].contiguous()
    slots[700:705], slots[2000:2100] = -1, slots[2000:2100].flip(0)
    bias = normal(vectors * dim) if options.get("bias") else None
    weights = [normal(dim) if options.get("weights") else None for _ in "qk"]
    angles = normal(n, rot // 2, 2) if rot else None
    def run(step):
        kept = [torch.full(shape(pages, kv_heads, page, -(-dim // 16) * 16), 7.0, dtype=torch.bfloat16, device=DEVICE) for shape in (key_page_shape, value_page_shape)]
        queries = [k.qk_norm_store(rows[i:i + step], *weights, 1e-6, positions[i:i + step], slots[i:i + step], 0.5 if options.get("temperature") else 0.0, 64, *kept, heads,
                                   kv_heads, dim, dim, torch.bfloat16, tiled_page_size=page if not alone else 0, bias=bias, normed=True, queries_only=alone,
                                   cos_sin=angles[i:i + step] if rot else None, values_normed=options.get("values_normed", False),
                                   norm_turned=options.get("norm_turned", False)) for i in range(0, n, step)]
        return [torch.cat(queries), *kept]
    for whole, parts in zip(run(n), run(125)):
        assert torch.equal(whole, parts)


@pytest.mark.parametrize("n,dtype", [(50, torch.float32), (50, torch.bfloat16), (9000, torch.bfloat16)])      # a wave a head, and eight tokens a wave
@pytest.mark.parametrize("norm_turned", [False, True])
def test_heads_norms_are_summed_in_one_order_with_the_same_roundings(n, dtype, norm_turned):
    """The bits of a head's norm, spelled out: a lane takes every 64th channel in order, by one multiply-add each, where the norm is that of turned vectors by
    a rounded square and an addition, in turned channels as in the others (of turned ones the square is multiplied by their length, here 1); lanes 32 apart
    meet first, neighbours last. No tolerance: every step is one rounding."""
    heads, kv_heads, dim, rot, eps = 3, 1, 192, 64, 1e-6
    vectors = heads + 2 * kv_heads
    assert (-(-n // 8) * vectors >= 4096) == (n == 9000)
    generator = torch.Generator(device=DEVICE).manual_seed(n + norm_turned)
    rows = torch.randn(n, vectors * dim, generator=generator, device=DEVICE)
    angles = torch.tensor([1.0, 0.0], device=DEVICE).repeat(n, rot // 2, 1).contiguous()       # no turn, so that the length is 1 and the turn changes no bit
    pages = -(-n // 16)
    slots = torch.arange(n, dtype=torch.int32, device=DEVICE)
    tiled = 16 if dtype == torch.bfloat16 else 0
    kept = ([torch.zeros(shape(pages, kv_heads, 16, dim), dtype=dtype, device=DEVICE) for shape in (key_page_shape, value_page_shape)] if tiled else
            [torch.zeros(pages, 16, kv_heads, dim, dtype=dtype, device=DEVICE) for _ in "kv"])
    q = kernels().qk_norm_store(rows, None, None, eps, slots, slots, 0.0, 1, *kept, heads, kv_heads, dim, dim, dtype, tiled_page_size=tiled, normed=True,
                                cos_sin=angles, norm_turned=norm_turned)
    x = rows.cpu().numpy().reshape(n, vectors, dim // 64, 64)[:, :heads]
    sums = np.zeros((n, heads, 64), np.float32)
    for j in range(dim // 64):
        square = x[:, :, j].astype(np.float64) ** 2                 # exact
        sums = (sums + square.astype(np.float32) if norm_turned else (sums + square)).astype(np.float32)
    for distance in (32, 16, 8, 4, 2, 1):
        sums = sums + sums[:, :, np.arange(64) ^ distance]
    factor = np.float32(1.0) / np.sqrt(sums[:, :, :1] / np.float32(dim) + np.float32(eps))
    want = torch.from_numpy(x.reshape(n, heads, dim) * factor).to(dtype).view(n, heads * dim)
    assert torch.equal(q.view(n, heads * dim).cpu(), want)


# ---- float32 attention by chunks, all heads of a kv head together: every head size, one head a kv head to more than 16, windows that begin in
# either tile of a chunk, and values that are not finite where a token sees them and where it does not ----
@pytest.mark.parametrize("heads,kv_heads,hd,page_size", [(28, 4, 16, 16), (14, 2, 32, 32), (9, 9, 48, 48), (7, 1, 64, 16), (40, 2, 80, 48), (5, 1, 96, 16),
                                                         (34, 2, 112, 32), (4, 1, 128, 16)])
@pytest.mark.parametrize("window", [0, 70, 190])
def test_chunks_for_all_heads_have_the_bits_of_a_wave_a_row(heads, kv_heads, hd, page_size, window):
    k, rng = kernels(), np.random.default_rng(hd + window)
    lengths, counts = [300, 1, 64, 65, 128, 129, 700, 193], [1, 1, 3, 1, 1, 2, 4, 1]
    t, *_ = build_paged_case(rng, torch.float32, lengths, counts, heads, kv_heads, hd, page_size)
    for broken in (None, float("nan"), float("inf")):
        if broken is not None:
            t["v"].view(-1)[::997] = broken
        run = lambda **way: k.paged_attention_rowwise(t["q"], t["k"], t["v"], t["table"], t["seq"], t["pos"], hd ** -0.5, window, heads, kv_heads, hd, **way)
        by_chunks, by_rows = run(split=True), run(split=False)
        assert torch.equal(torch.nan_to_num(by_chunks, 7.0, 8.0, 9.0), torch.nan_to_num(by_rows, 7.0, 8.0, 9.0)), broken



# Both sides of each line between the kernel for all heads and a wave a head (24, 64, 128 and 256 keys; 320 to 8192 workgroups), single tokens and portions
@pytest.mark.parametrize("heads,kv_heads,hd", [(8, 8, 128), (12, 12, 48), (4, 2, 64), (9, 3, 16), (28, 4, 32)])
@pytest.mark.parametrize("requests,portion,lengths", [(41, 1, (24, 25)), (81, 1, (40, 64, 65)), (100, 1, (128, 129)), (60, 1, (256, 600)), (2, 5, (24, 25)), (4, 20, (64, 65)),
                                                       (1, 70, (128, 129)), (1, 48, (300, 600)), (3, 30, (1100,))])
def test_chunks_have_the_same_bits_whichever_kernel_takes_them(heads, kv_heads, hd, requests, portion, lengths):
    k = kernels()
    for length in lengths:
        rng = np.random.default_rng(length + hd)
        t, *_ = build_paged_case(rng, torch.float32, [length] * requests, [min(portion, length)] * requests, heads, kv_heads, hd, 16)
        run = lambda **way: k.paged_attention_rowwise(t["q"], t["k"], t["v"], t["table"], t["seq"], t["pos"], hd ** -0.5, 0, heads, kv_heads, hd, longest=2048,
                                                      usual=length, **way)
        by_rows = run(split=False)
        assert torch.equal(run(split=True), by_rows) and torch.equal(run(), by_rows), length



def test_a_step_that_can_go_without_a_workspace_does_where_there_is_no_room(monkeypatch):
    k, rng = kernels(), np.random.default_rng(3)
    heads, kv_heads, hd = 28, 4, 32
    allocate = torch.empty

    def full(*sizes, **options):
        if sizes and isinstance(sizes[0], tuple) and len(sizes[0]) == 4:      # the chunks' results
            raise torch.OutOfMemoryError("no room")
        return allocate(*sizes, **options)

    for requests in (80, 20):       # 2240 rows, and 560, which always had a workspace
        t, *_ = build_paged_case(rng, torch.float32, [300] * requests, [1] * requests, heads, kv_heads, hd, 16)
        run = lambda: k.paged_attention_rowwise(t["q"], t["k"], t["v"], t["table"], t["seq"], t["pos"], hd ** -0.5, 0, heads, kv_heads, hd)
        want = run()
        with monkeypatch.context() as patch:
            patch.setattr(torch, "empty", full)
            if requests == 80:
                assert torch.equal(run(), want)
            else:
                with pytest.raises(torch.OutOfMemoryError):
                    run()


# ---- gates of every size: where exp(-gate) leaves the numbers the quotient is the gate or nothing, in every kernel that forms one ----
GATES = [-1.0, -20.0, -86.5, -87.5, -90.0, -100.0, -1e3, -1e13, -1e30, -3.3895313892515355e38, 1.0, 87.5, 1e3, 1e13, 1e30, 3.3895313892515355e38]
CLAMP, SLOPE = 7.0, 1.702


def gated_in_64_bits(gate, up, kind):
    """``gate * sigmoid(t) * up`` without a step that leaves the numbers; at -inf it is no number, as -inf * 0 is."""
    gate, up = np.asarray(gate, np.float64), np.asarray(up, np.float64)
    if kind == "clamped":
        gate, up = np.minimum(gate, CLAMP), np.clip(up, -CLAMP, CLAMP) + 1.0
    t = {"silu": gate, "gelu_tanh": math.sqrt(8.0 / math.pi) * (gate + 0.044715 * gate ** 3), "clamped": SLOPE * gate}[kind]
    small = np.exp(-np.abs(t))
    with np.errstate(invalid="ignore"):
        return gate * (np.where(t < 0, small, 1.0) / (1.0 + small)) * up


def assert_gated(got, gate, up, kind):
    """A rounding to bfloat16 and a little, or below its smallest normal number."""
    gate, up = (torch.tensor(values).to(torch.bfloat16).double().numpy() for values in (gate, up))
    want = np.broadcast_to(gated_in_64_bits(gate, up, kind), got.shape)
    np.testing.assert_allclose(got.double().cpu().numpy(), want, rtol=2.0 ** -8, atol=2.0 ** -126)


@pytest.mark.parametrize("kind", ["silu", "gelu_tanh"])
@pytest.mark.parametrize("shift", [0, 1])       # rows that begin at a 16-byte boundary or not
def test_activations_of_gates_of_every_size(kind, shift):
    gates = GATES + [float("-inf"), float("inf"), float("nan")] + [-0.0] * 5
    ups = [0.5, -0.25] * (len(gates) // 2)
    rows = torch.empty(3 * 2 * len(gates) + shift, dtype=torch.bfloat16, device=DEVICE)[shift:].view(3, 2 * len(gates))
    rows.copy_(torch.tensor(gates + ups))
    assert_gated(kernels().gated_activation(rows, kind), gates, ups, kind)


@pytest.mark.parametrize("product,rows,kind", [(product, rows, kind) for product, rows in (("skinny", 5), ("skinny", 16), ("medium", 40), ("tiled", 130))
                                                for kind in ("silu", "gelu_tanh", "clamped") if (product, kind) != ("medium", "clamped")])
@pytest.mark.parametrize("width", [16, 13])     # whole pieces of 16 bytes of results, and not
def test_products_with_gates_of_every_size(product, rows, kind, width):
    k, gates, ups = kernels(), GATES[:width], ([0.5, -0.25] * 8)[:width]
    x, weight = torch.zeros((rows, 64), dtype=torch.bfloat16, device=DEVICE), torch.zeros((2 * width, 64), dtype=torch.bfloat16, device=DEVICE)
    x[:, 40], weight[:, 40] = 1.0, torch.tensor(gates + ups, device=DEVICE)      # so that the sums are the gates themselves
    packed = k.pack_weight(weight, interleave_halves=True)
    if kind == "clamped":
        got = k.gemm_skinny_clamped(x, packed, 2 * width, CLAMP, SLOPE) if product == "skinny" else k.gemm_tiled(x, packed, 2 * width, "clamped", limit=CLAMP, slope=SLOPE)
    else:
        got = {"skinny": k.gemm_skinny, "medium": k.gemm_medium, "tiled": k.gemm_tiled}[product](x, packed, 2 * width, "gated" if kind == "silu" else "gated_gelu")
    assert_gated(got, gates, ups, kind)


@pytest.mark.parametrize("tokens,grouped", [(4, False), (60, True), (700, True)])       # few pairs on the matrix units, tiles of pairs, large tiles
@pytest.mark.parametrize("kind", ["silu", "clamped"])
def test_experts_with_gates_of_every_size(tokens, grouped, kind):
    k, size, gates, ups = kernels(), 512, GATES * 32, [0.5, -0.25] * 256
    x, gate_up = torch.zeros((tokens, size), dtype=torch.bfloat16, device=DEVICE), torch.zeros((2, 2 * size, size), dtype=torch.bfloat16, device=DEVICE)
    x[:, 40], gate_up[:, :, 40] = 1.0, torch.tensor(gates + ups, device=DEVICE)
    down = torch.eye(size, device=DEVICE).to(torch.bfloat16).repeat(2, 1, 1)       # the result is the inner values
    ids, weights = (torch.arange(tokens, device=DEVICE, dtype=torch.int32) % 2)[:, None].contiguous(), torch.ones((tokens, 1), device=DEVICE)
    options = dict(activation="clamped_glu", limit=CLAMP, slope=SLOPE) if kind == "clamped" else {}
    assert_gated(k.moe_experts(x, ids, weights, gate_up, down, False, grouped=grouped, **options)[0], gates, ups, kind)


@pytest.mark.parametrize("vocab", [1, 63, 2048, 131072, 163840, 163841, 196608, 196609, 330000])
def test_tokens_of_vocabularies_up_to_and_beyond_what_a_thread_asks_for_at_once(vocab):
    """Ten logits of a slice a thread and twelve of a piece: one more, and the loops go round again. Top-k against torch's, ends of the range of draws."""
    k, generator = kernels(), torch.Generator(device=DEVICE).manual_seed(vocab)
    logits = torch.randn((6, vocab), generator=generator, device=DEVICE)
    logits[1, vocab - 1] = 9.0                      # the last token of all is the first maximum
    logits[2] = logits[2].round()                   # ties at the k-th value
    top = min(vocab, 30)
    values = torch.tensor([[0.8, 0.0, 0.7, 1.0, 0.9, 1.1], [0.0, 0.5, 0.999999, 0.5, 0.999999, 0.0]], device=DEVICE)
    chosen = k.sample(logits, values[0], torch.tensor([top, 0, top, 1, 0, 0], dtype=torch.int32, device=DEVICE), values[1]).tolist()
    assert chosen[1] == vocab - 1 and chosen[3] == int(logits[3].argmax()) and chosen[5] == 0 and chosen[4] > vocab - 1 - max(2, vocab // 100)
    for row, first in ((0, True), (2, False)):      # the lowest ids among those that equal the k-th value
        kept = sorted(torch.sort(logits[row], descending=True, stable=True).indices[:top].tolist())
        assert chosen[row] in (kept[:2] if first else kept[-2:])
    assert k.argmax(logits).tolist() == logits.argmax(1).tolist()
    logits[4, vocab // 2] = float("inf")
    assert k.argmax(logits)[4] == -1 and k.sample(logits, values[0], None, values[1])[4] == -1


@pytest.mark.parametrize("words", [1, 2, 3])
def test_the_scratch_of_a_draw_begins_at_any_word(words):
    """It is promised four bytes of alignment, not the sixteen that a load of four words takes: the same tokens from every word on."""
    k, lib, generator = kernels(), library.load(), torch.Generator(device=DEVICE).manual_seed(words)
    rows, vocab = 7, 9001
    logits, uniform = torch.randn((rows, vocab), generator=generator, device=DEVICE), torch.rand(rows, generator=generator, device=DEVICE)
    temperature, top_k = torch.full((rows,), 0.9, device=DEVICE), torch.tensor([0, 1, 40, 3000, 0, 2, 9001], dtype=torch.int32, device=DEVICE)
    scratch, out = torch.empty(lib.mll_sample_workspace(rows, vocab) // 4 + words, dtype=torch.int32, device=DEVICE), torch.empty(rows, dtype=torch.int32, device=DEVICE)
    for restricted in (top_k, None):
        k._check(lib.mll_sample(k._ptr(logits), k._ptr(temperature), k._ptr(restricted), k._ptr(uniform), k._ptr(out), k._ptr(scratch[words:]), rows, vocab, k._stream()), lib)
        assert torch.equal(out, k.sample(logits, temperature, restricted, uniform))


def test_the_best_tokens_of_the_longest_vocabulary():
    """2^31 - 2048 logits (8.6 GB): what a thread asks for behind the last one lies beyond 2^31. Two thirds of the weight are the last token's."""
    if torch.cuda.mem_get_info()[0] < 12 << 30:
        pytest.skip("needs 12 GB")
    vocab = 2 ** 31 - 2048
    logits = torch.full((1, vocab), -3.0, device=DEVICE)
    logits[0, vocab - 1], logits[0, 5] = math.log(2.0), 0.0
    one = torch.ones(1, device=DEVICE)
    chosen = [int(kernels().sample(logits, one, torch.full((1,), top, dtype=torch.int32, device=DEVICE), draw * one)) for top in (2, 1) for draw in (0.0, 0.3, 0.4, 0.99)]
    assert chosen == [5, 5, vocab - 1, vocab - 1] + [vocab - 1] * 4


@pytest.mark.parametrize("m", [17, 32, 33, 48, 49, 64])
@pytest.mark.parametrize("n,k,splits", [(40, 8, 1), (300, 40, 1), (260, 264, 2), (1000, 1032, 3), (4112, 520, 1), (200, 2312, 4)])
def test_activations_that_are_not_finite_stay_in_their_row(m, n, k, splits):
    """Reductions that end within a k step, within a pair of them and within a stage: what lies behind a row's end is the next row, all of it NaN here."""
    ka, generator = kernels(), torch.Generator(device=DEVICE).manual_seed(m + n + k)
    x, w = ((torch.randn(shape, generator=generator, device=DEVICE) * scale).to(torch.bfloat16) for shape, scale in (((m, k), 1.0), ((n, k), k ** -0.5)))
    packed, spoilt = ka.pack_weight(w), x.clone()
    spoilt[1::2] = float("nan")
    spoilt[m - 1] = float("inf") if m % 2 == 1 else float("nan")
    for plan in ((2, 8, splits), (1, 4, splits)):
        whole = ka.gemm_medium(x, packed, n, "f32", plan=plan)
        got = ka.gemm_medium(spoilt, packed, n, "f32", plan=plan)
        kept = [row for row in range(0, m - 1, 2)]
        assert torch.equal(got[..., kept, :], whole[..., kept, :])
        total = whole.sum(0) if splits > 1 else whole
        assert float((total - x.float() @ w.float().T).abs().max()) < 2e-6 * k ** 0.5 + 1e-5      # k products of size 1 / sqrt(k)
        assert not got[..., 1, :].isfinite().any() if splits == 1 else not got.sum(0)[1].isfinite().any()


@pytest.mark.parametrize("rows", [41, 64])
def test_wide_products_of_41_to_64_rows_at_any_address(rows):
    """A head's weight by the packed copy, and by the library where the rows begin at no 16-byte boundary: float32 sums of 512 products of size
    1 / sqrt(512) in two orders."""
    from microllm_rocm_amd.parts.linear import Weight, linear, takes_packed
    generator = torch.Generator(device=DEVICE).manual_seed(rows)
    n, k = 32768, 512
    x, w = ((torch.randn(shape, generator=generator, device=DEVICE) * scale).to(torch.bfloat16) for shape, scale in (((rows, k), 1.0), ((n, k), k ** -0.5)))
    weight = Weight(w)
    apart = torch.empty(rows * k + 1, dtype=torch.bfloat16, device=DEVICE)[1:].view(rows, k)
    apart.copy_(x)
    assert takes_packed(weight, rows, address=x.data_ptr()) and not takes_packed(weight, rows, address=apart.data_ptr())
    got, want = (linear(rows_, weight, out_dtype=torch.float32) for rows_ in (apart, x))
    assert float((got - want).abs().max()) < 2e-5


@pytest.mark.parametrize("width", [4, 252, 896, 1028, 4096])
@pytest.mark.parametrize("parts", [1, 2, 4, 8, 16])
def test_norms_of_few_rows_have_the_bits_of_any_number_of_parts(width, parts):
    """The kernel that asks for all parts at once against the one for any number, which parts of zeros lead to: the same additions."""
    k, generator = kernels(), torch.Generator(device=DEVICE).manual_seed(width + parts)
    draw = lambda *shape: torch.randn(shape, generator=generator, device=DEVICE)
    h, weight, delta = draw(5, width), draw(width), draw(parts, 5, width)
    more = torch.cat([delta, torch.zeros((1 if parts > 1 else 2, 5, width), device=DEVICE)])      # 3, 3, 5, 9 and 17
    rows = torch.tensor([4, 0, 2], dtype=torch.int32, device=DEVICE)
    for dtype in (torch.bfloat16, torch.float32):
        for options in (dict(write_h=True), dict(rows=rows)):
            streams, results = (h.clone(), h.clone()), []
            for stream, given in zip(streams, (delta if parts > 1 else delta[0], more)):
                results.append(k.rms_norm(stream, weight, 1e-6, dtype, delta=given, **options))
            assert torch.equal(*results) and torch.equal(*streams)
        alone = k.rms_norm(h, weight, 1e-6, dtype)
        assert torch.equal(alone, k.rms_norm(h, weight, 1e-6, dtype, delta=torch.zeros((3, 5, width), device=DEVICE)))
    v = h.double() + delta.double().sum(0)
    want = v / torch.sqrt((v * v).mean(1, keepdim=True) + 1e-6) * weight.double()
    got = k.rms_norm(h, weight, 1e-6, torch.float32, delta=delta if parts > 1 else delta[0])
    assert float((got - want).norm() / want.norm()) < 4e-7 * parts ** 0.5      # parts + 1 additions of numbers rounded to 2^-24


@pytest.mark.parametrize("heads,kv_heads,hd,page_size", [(14, 2, 64, 16), (3, 1, 16, 32), (5, 5, 48, 16), (28, 4, 128, 16), (2, 0, 256, 16)])
@pytest.mark.parametrize("parts,biased", [(1, True), (2, False), (4, True), (8, True), (16, True)])
def test_queries_keys_and_values_in_pairs_have_the_bits_of_any_number_of_parts(heads, kv_heads, hd, page_size, parts, biased):
    """Two pairs or four dims a thread against the kernel for any number of parts, which parts of zeros lead to; tokens without a place in a page among them."""
    k, generator = kernels(), torch.Generator(device=DEVICE).manual_seed(heads + hd + parts)
    tokens, total = 19, (heads + 2 * kv_heads) * hd
    draw = lambda *shape: torch.randn(shape, generator=generator, device=DEVICE)
    qkv, bias = draw(parts, tokens, total), draw(total) if biased else None
    angle = draw(tokens, hd // 2)
    cos_sin = torch.stack([angle.cos(), angle.sin()], dim=2).contiguous()
    slots = (torch.randperm(3 * page_size, generator=generator, device=DEVICE)[:tokens]).to(torch.int32)
    slots[[2, 11]] = -1
    pos, results = torch.arange(tokens, device=DEVICE, dtype=torch.int32), []
    for given in (qkv if parts > 1 else qkv[0], torch.cat([qkv, torch.zeros((1 if parts > 1 else 2, tokens, total), device=DEVICE)])):
        pages = [torch.full(shape(3, max(kv_heads, 1), page_size, hd), 5.0, dtype=torch.bfloat16, device=DEVICE) for shape in (key_page_shape, value_page_shape)]
        stored = (slots, None, *pages) if kv_heads else (None, None, None, None)
        q = k.qkv_rope_store(given, bias, pos, *stored, heads, kv_heads, hd, page_size, torch.bfloat16, pair_order=True, cos_sin=cos_sin)
        results.append([q, *pages])
    assert all(torch.equal(a, b) for a, b in zip(*results))


@pytest.mark.parametrize("splits", [2, 8, 9, 17])
def test_joined_splits_of_a_step_padded_to_a_fixed_length(splits):
    """Eight splits are asked for before an entry's token is known, whatever it is: none of a padded list's other rows is written."""
    rng, heads, kv_heads, hd = np.random.default_rng(splits), 6, 2, 80
    lengths = [517, 1, 33, 960, 40, 7]
    t, q_exact, ek, ev, seq, pos = build_paged_case(rng, torch.bfloat16, lengths, [1] * len(lengths), heads, kv_heads, hd, 16)
    some = torch.tensor([3, -1, 0, -1, -1, 1], dtype=torch.int32, device=DEVICE)
    out = torch.full_like(t["q"], 7.0)
    kernels().paged_attention_decode(t["q"], t["k"], t["v"], t["table"], t["seq"], t["pos"], hd ** -0.5, 0, heads, kv_heads, hd, splits, out=out, token_ids=some)
    want = reference_attention(q_exact, ek, ev, seq, pos, heads, kv_heads, hd, hd ** -0.5, 0)
    np.testing.assert_allclose(out.float().cpu().numpy()[[0, 1, 3]], want[[0, 1, 3]], **tolerance(torch.bfloat16))
    assert bool((out[[2, 4, 5]] == 7.0).all())


@pytest.mark.parametrize("heads,kv_heads,hd,page_size,tokens", [(14, 2, 64, 16, 65), (3, 1, 16, 32, 72), (5, 5, 48, 16, 71), (28, 4, 128, 16, 130), (2, 0, 256, 16, 66), (2, 1, 80, 48, 200)])
@pytest.mark.parametrize("parts,dtype", [(1, torch.bfloat16), (3, torch.bfloat16), (1, torch.float32)])
def test_queries_keys_and_values_of_eight_tokens_a_wave_have_the_bits_of_a_block_a_token(heads, kv_heads, hd, page_size, tokens, parts, dtype):
    """More than 64 tokens against the same tokens 64 at a time, which another kernel takes: tokens beyond the last eight, items beyond a block's, places in any order
    and tokens without one."""
    k, generator = kernels(), torch.Generator(device=DEVICE).manual_seed(heads + hd + tokens)
    total, pages = (heads + 2 * kv_heads) * hd, -(-tokens // page_size) + 1
    draw = lambda *shape: torch.randn(shape, generator=generator, device=DEVICE)
    qkv, bias, angle = draw(parts, tokens, total), draw(total), draw(tokens, hd // 2)
    cos_sin = torch.stack([angle.cos(), angle.sin()], dim=2).contiguous()
    slots = torch.arange(tokens, device=DEVICE, dtype=torch.int32) + 3
    slots[20:60] = slots[20:60].flip(0)
    slots[[2, tokens - 1]] = -1
    pos, results = torch.arange(tokens, device=DEVICE, dtype=torch.int32), []
    for step in (tokens, 64):
        stored = [torch.full(shape(pages, max(kv_heads, 1), page_size, hd), 5.0, dtype=dtype, device=DEVICE) for shape in (key_page_shape, value_page_shape)]
        q = []
        for first in range(0, tokens, step):
            rows = slice(first, min(first + step, tokens))
            given = qkv[:, rows].contiguous() if parts > 1 else qkv[0, rows]
            places = (slots[rows], None, *stored) if kv_heads else (None, None, None, None)
            q.append(k.qkv_rope_store(given, bias, pos[rows], *places, heads, kv_heads, hd, page_size, dtype, cos_sin=cos_sin[rows]))
        results.append([torch.cat(q), *stored])
    assert all(torch.equal(a, b) for a, b in zip(*results))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("width,offset", [(4, 0), (252, 0), (3584, 0), (4100, 0), (896, 1), (1002, 0)])
def test_embedding_rows_of_every_width_and_address(width, offset, dtype):
    """Four columns a thread, in one round and in two, and the rows that begin at no whole four of them; ids outside the table."""
    generator = torch.Generator(device=DEVICE).manual_seed(width)
    flat = torch.randn(37 * width + offset, generator=generator, device=DEVICE).to(dtype)
    table, ids = flat[offset:].view(37, width), torch.tensor([36, 0, -1, 5, 37, 5], dtype=torch.int32, device=DEVICE)
    out = kernels().embedding(table, ids, scale=1.5)
    known = [0, 1, 3, 5]
    assert torch.equal(out[known], table[ids[known].long()].float() * 1.5) and bool(out[[2, 4]].isnan().all())


@pytest.mark.parametrize("width", [1, 2, 129, 2048, 2051])
def test_position_waves_of_every_width(width):
    """Two columns a thread: the last one alone, one round and two, ids outside the table. One rounding of the wave (2^-24 at most) and one of the sum."""
    generator = torch.Generator(device=DEVICE).manual_seed(width)
    table = torch.randn((11, width), generator=generator, device=DEVICE)
    ids, pos = torch.tensor([10, 0, -1, 11, 3], dtype=torch.int32, device=DEVICE), torch.tensor([0, 1, 5, 7, 31999], dtype=torch.int32, device=DEVICE)
    rates = 10000.0 ** (-torch.arange((width + 1) // 2, dtype=torch.float64, device=DEVICE) * 2 / width)
    got = kernels().embedding_sinusoid(table, ids, pos, rates)
    angle = (pos.double()[:, None] * rates).repeat_interleave(2, 1)[:, :width]
    wave = torch.where(torch.arange(width, device=DEVICE) % 2 == 0, angle.sin(), angle.cos())
    want = table[ids.clamp(0, 10).long()].double() + wave
    assert bool(got[[2, 3]].isnan().all())
    assert float((got - want)[[0, 1, 4]].abs().max()) <= 2 ** -24 * (1 + float(want.abs().max()))


@pytest.mark.parametrize("value_dim", [1, 63, 64, 65, 128, 200, 256, 257])
@pytest.mark.parametrize("weighted", [False, True])
def test_gated_heads_of_every_size(value_dim, weighted):
    """One, two and four values a lane, and those a wave does not hold; a row a workgroup and four, the last of which have none, with the same bits."""
    k, generator = kernels(), torch.Generator(device=DEVICE).manual_seed(value_dim)
    heads, tokens, before = 3, 701, 5
    draw = lambda *shape: torch.randn(shape, generator=generator, device=DEVICE)
    o, proj, weight = draw(tokens, heads * value_dim), draw(tokens, before + heads * value_dim + 2), draw(value_dim) if weighted else None
    run = lambda rows: k.gla_gate(o[:rows], proj[:rows], before, weight, 1e-5, heads, value_dim, 1.5, torch.float32)
    got = run(tokens)
    assert torch.equal(got[:7], run(7))
    v, g = o.double().view(tokens, heads, value_dim), proj[:, before:before + heads * value_dim].double().view(tokens, heads, value_dim)
    want = v / torch.sqrt((v * v).mean(2, keepdim=True) + 1e-5) * (weight.double() if weighted else 1.0) * g * torch.sigmoid(g) * 1.5
    assert float((got.double().view_as(want) - want).norm() / want.norm()) < 1e-6      # some ten roundings of 2^-24


@pytest.mark.parametrize("dtype", [np.float32, np.int64])
def test_uploads_hold_what_was_given_while_the_device_is_busy(dtype):
    """The host goes on, writes over its array and gives the pinned copies back before the device has read any: a hundred uploads of some sizes behind 50 ms and
    more of other work, from arrays in any order of their dims."""
    from microllm_rocm_amd.ops.transfers import on_device_later
    target = torch.device(DEVICE)
    shapes = [(3, 97), (1,), (2, 0), (5, 4)]
    for busy in (False, True):      # the first round makes the pinned memory, which may wait
        torch.cuda.synchronize()
        done, got = torch.cuda.Event(), []
        if busy:
            torch.cuda._sleep(100_000_000)
        done.record()
        for number in range(100):
            rows, columns = (shapes[number % 4] + (1,))[:2]
            array = np.empty((columns, rows), dtype=dtype).T
            array[...] = number + np.arange(rows * columns).reshape(rows, columns) / 1
            got.append(on_device_later(array, target))
            array[...] = -1
        assert not busy or not done.query()
        for number, tensor in enumerate(got):
            rows, columns = (shapes[number % 4] + (1,))[:2]
            assert tensor.device.type == "cuda" and tensor.cpu().tolist() == (number + np.arange(rows * columns).reshape(rows, columns)).tolist()
