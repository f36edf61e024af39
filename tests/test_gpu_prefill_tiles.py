"""The chunked-prefill kernel against the float64 oracle where its tiles can go wrong: chunk
lengths around the 128-column tile and the 32-key half steps, histories that end inside a
block, columns scaled out of f16's range, key factors past the safe range of scores, V
scales of very different exponents in one step, and id windows past 64 steps."""

import numpy as np
import pytest
import torch

from aster_amd import KVQuantization, PagedKVCache
from aster_amd.attention_backend import UnsupportedAttentionBackend
from tests.gpu_util import mark_padding, oracle_decode

pytestmark = pytest.mark.gpu


def _cache(device, rows, dim, kv, fmt, seed):
    """Random codes and scales under shuffled tables for contexts ``rows``."""
    gen = torch.Generator(device=device).manual_seed(seed)
    pages = [-(-n // 16) for n in rows]
    perm = np.random.default_rng(seed).permutation(sum(pages) + 2).astype(np.int32)
    tables = np.zeros((len(rows), max(pages)), np.int32)
    at = 0
    for row, n in enumerate(pages):
        tables[row, :n] = perm[at:at + n]
        at += n
    cache = PagedKVCache(num_blocks=len(perm), num_layers=1, num_kv_heads=kv, head_dim=dim,
                         device=device, quantization=KVQuantization(fmt))
    x = torch.randn(cache.codes.shape, generator=gen, device=device)
    most = {"int8": 127.0, "fp8_e4m3fn": 448.0, "fp8_e5m2": 57344.0}[fmt]
    amax = x.abs().amax(-1)
    units = x / amax[..., None] * most
    codes = units.round() if fmt == "int8" else units
    cache.codes.copy_(codes.to(cache.quantization.dtype).view(torch.int8))
    cache.scales.copy_(amax / most)
    return cache, tables, gen


def _check(cache, tables, lens, counts, query, window=None, atol=2e-3, rtol=2e-3, bound=None,
           causal=True, **options):
    device = query.device
    starts = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    out = cache.paged_attention(0, query, torch.from_numpy(tables).to(device),
                                torch.from_numpy(np.array(lens, np.int32)).to(device),
                                max_context_len=bound or max(lens), window=window,
                                query_start_loc=torch.from_numpy(starts).to(device),
                                max_query_len=max(counts), causal=causal, check=True, **options)
    want = oracle_decode(tables, cache, query, context_lens=np.array(lens, np.int32),
                         scale=cache.head_dim ** -0.5, window=window, causal=causal,
                         query_lens=np.array(counts, np.int32), fp64=True)
    bf16 = query.dtype == torch.bfloat16  # outputs rounded to 2^-9 of themselves
    np.testing.assert_allclose(out.float().cpu().numpy(), want, atol=atol,
                               rtol=5e-3 if bf16 else rtol)


@pytest.mark.parametrize("fmt", ["int8", "fp8_e4m3fn", "fp8_e5m2"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("dim,kv,group", [(64, 2, 4), (128, 2, 1), (128, 1, 16), (256, 2, 2)])
def test_tile_edges(device, dim, kv, group, dtype, fmt):
    tile = 128 // group
    counts = [2, tile - 1 if tile > 2 else 3, tile, tile + 1, 2 * tile + 5]
    priors = [0, 31, 32, 33, 64]
    lens = [n + p for n, p in zip(counts, priors)]
    cache, tables, gen = _cache(device, lens, dim, kv, fmt, dim + group)
    query = torch.randn((sum(counts), kv * group, dim), generator=gen, device=device).to(dtype)
    _check(cache, tables, lens, counts, query)
    _check(cache, tables, lens, counts, query, window=37)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("power", [-70, -40, -14, -9, -4, 13])
def test_scaled_columns(device, dtype, power):
    """Queries whose columns leave the unscaled range beside zero ones, in prompt and history
    keys; key scales of 2^-power keep the scores ordinary."""
    if dtype == torch.float16 and power < -9:
        pytest.skip("outside fp16")
    lens, counts = [100, 350], [40, 17]
    cache, tables, gen = _cache(device, lens, 128, 2, "int8", 7)
    query = torch.randn((sum(counts), 8, 128), generator=gen, device=device) * 2.0 ** power
    query[:, 1::2] = 0
    cache.scales[:, :, 0] *= 2.0 ** -power
    _check(cache, tables, lens, counts, query.to(dtype))


@pytest.mark.parametrize("fmt", ["int8", "fp8_e4m3fn", "fp8_e5m2"])
def test_large_scales(device, fmt):
    """V scales up to 2^20 larger in some blocks, beside ordinary ones: no product or sum
    leaves its range. The tolerance is of the largest values (the weights' f16 rounding), so
    that only these blocks are checked here; test_exponents_of_padded_blocks has the others'."""
    lens, counts = [300, 90], [70, 33]
    cache, tables, gen = _cache(device, lens, 128, 2, fmt, 11)
    cache.scales[::3, :, 1] *= 2.0 ** 20
    cache.scales[1::6, :, 1] *= 2.0 ** 11
    query = torch.randn((sum(counts), 8, 128), generator=gen, device=device).half().float()
    _check(cache, tables, lens, counts, query, atol=2.0 ** 20 * 2e-3)


def test_overflowing_scores_raise(device):
    lens, counts = [80], [40]
    cache, tables, gen = _cache(device, lens, 128, 1, "int8", 3)
    cache.scales[int(tables[0, 1]), 0, 0] = 3e37
    query = 1e3 * torch.randn((40, 4, 128), generator=gen, device=device)
    with pytest.raises(ValueError, match="overflow"):
        _check(cache, tables, lens, counts, query)


@pytest.mark.parametrize("fmt", ["int8", "fp8_e4m3fn"])
@pytest.mark.parametrize("slot", [0, 70, 79])
def test_nan_key_scale(device, fmt, slot):
    """A NaN key scale is reported where a query sees its key, and nowhere else: past the
    context (the block's last slot) it changes nothing."""
    lens, counts = [79], [40]
    cache, tables, gen = _cache(device, lens, 128, 1, fmt, 3)
    query = torch.randn((40, 4, 128), generator=gen, device=device).bfloat16()
    cache.scales[int(tables[0, slot // 16]), 0, 0, 0, slot % 16] = float("nan")
    if slot < 79:
        with pytest.raises(ValueError, match="overflow"):
            _check(cache, tables, lens, counts, query)
    else:
        _check(cache, tables, lens, counts, query)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_smallest_key_scales(device, dtype):
    """Key scales at the quantizer's least (the smallest normal number) under queries large
    enough for ordinary scores: their factor is below the normal range, which costs it
    2^-21 of itself."""
    lens, counts = [79], [40]
    cache, tables, gen = _cache(device, lens, 128, 1, "int8", 3)
    cache.scales[:, :, 0] = 2.0 ** -126
    query = (torch.randn((40, 4, 128), generator=gen, device=device) * 2.0 ** 119).to(dtype)
    _check(cache, tables, lens, counts, query)


def test_long_history(device):
    """A unit of 130 key steps, its ids read one step ahead of its blocks, in a window too."""
    lens, counts = [64 * 64 * 2 + 77], [9]
    cache, tables, gen = _cache(device, lens, 64, 1, "int8", 5)
    query = torch.randn((9, 2, 64), generator=gen, device=device).half()
    _check(cache, tables, lens, counts, query)
    _check(cache, tables, lens, counts, query, window=5000)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("dim,kv,group", [(128, 1, 4), (64, 2, 2), (256, 1, 8)])
@pytest.mark.parametrize("counts,priors", [([5], [3000]), ([40, 33], [2500, 100]),
                                           ([129, 2, 60], [1100, 2048, 0])])
def test_split_units(device, dim, kv, group, dtype, counts, priors):
    """Few units over long histories: cut into key ranges and merged, shorter units beside
    them whole, windows that leave a tile few keys, a history far below the declared bound."""
    lens = [n + p for n, p in zip(counts, priors)]
    cache, tables, gen = _cache(device, lens, dim, kv, "int8", dim)
    query = torch.randn((sum(counts), kv * group, dim), generator=gen, device=device).to(dtype)
    _check(cache, tables, lens, counts, query)
    _check(cache, tables, lens, counts, query, window=700)
    wide = np.zeros((len(lens), 2048), np.int32)
    wide[:, :tables.shape[1]] = tables
    _check(cache, wide, lens, counts, query, bound=16 * 2048)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_one_token_rows_beside_chunks(device, dtype):
    """Short contexts: the prefill launch serves the one-token rows (16-bit queries), an
    empty context included; equal chunks whose offsets hold a one-token row all the same."""
    counts, priors = [1, 30, 1, 1, 7], [100, 0, 0, 400, 33]
    lens = [n + p for n, p in zip(counts, priors)]
    cache, tables, gen = _cache(device, lens, 128, 2, "int8", 9)
    query = torch.randn((sum(counts), 8, 128), generator=gen, device=device).to(dtype)
    _check(cache, tables, lens, counts, query)
    lens[2] = 0
    _check(cache, tables, lens, counts, query)
    # 3 rows x 4 tokens declared, offsets that give 1 + 4 + 4
    starts = torch.tensor([0, 1, 5, 9], dtype=torch.int32, device=device)
    sub = torch.from_numpy(tables[:3]).to(device)
    ctx = torch.tensor([50, 30, 16], dtype=torch.int32, device=device)
    out = cache.paged_attention(0, query[:12], sub, ctx, max_context_len=64,
                                query_start_loc=starts, max_query_len=4, check=True)
    want = oracle_decode(tables[:3], cache, query[:9], context_lens=np.array([50, 30, 16], np.int32),
                         scale=128 ** -0.5, query_lens=np.array([1, 4, 4], np.int32), fp64=True)
    np.testing.assert_allclose(out[:9].float().cpu().numpy(), want, atol=2e-3, rtol=5e-3)
    if dtype == torch.float32:  # one-token rows in exact fp32: sums of 50 terms of order 1
        np.testing.assert_allclose(out[0].cpu().numpy(), want[0], atol=2e-5, rtol=0)


@pytest.mark.parametrize("counts", [[16], [16, 16], [16, 3]])
def test_group_of_16_at_head_dim_256_is_refused(device, counts):
    """16-bit queries in groups the decode kernels do not take, whatever the chunks' lengths."""
    lens = [n + 40 for n in counts]
    cache, tables, gen = _cache(device, lens, 256, 1, "int8", 3)
    query = torch.randn((sum(counts), 16, 256), generator=gen, device=device).bfloat16()
    with pytest.raises(UnsupportedAttentionBackend, match="group size 16"):
        _check(cache, tables, lens, counts, query)


def _two_groups(device, dim, fmt, n, first, codes, k_scale, v):
    """One chunk of 9 queries after ``n`` keys of one head: keys below ``first`` and the rest
    with K codes ``codes[0]`` and ``codes[1]`` in every dimension but the first (0 there), K
    scales ``k_scale[0]`` and ``[1]``, values ``v[0]`` and ``v[1]``."""
    cache, tables, _ = _cache(device, [n], dim, 1, fmt, 3)
    most = {"int8": 127.0, "fp8_e4m3fn": 448.0, "fp8_e5m2": 57344.0}[fmt]
    at = torch.arange(n, device=device)
    pages, slots = torch.from_numpy(tables[0]).to(device).long()[at // 16], at % 16
    pick = lambda pair: torch.where(at < first, float(pair[0]), float(pair[1]))
    code = lambda x: x.to(cache.quantization.dtype).view(torch.int8)
    cache.codes[pages, 0, 0, 0, slots] = code(pick(codes)[:, None].repeat(1, dim))
    cache.codes[pages, 0, 0, 0, slots, 0] = 0
    cache.codes[pages, 0, 1, 0, slots] = code(pick([most if x else 0 for x in v])[:, None].repeat(1, dim))
    cache.scales[pages, 0, 0, 0, slots] = pick(k_scale)
    cache.scales[pages, 0, 1, 0, slots] = pick([x / most if x else 1.0 for x in v])
    return cache, tables


@pytest.mark.parametrize("fmt,dim", [("int8", 128), ("fp8_e5m2", 256)])
@pytest.mark.parametrize("low", [-2e38, -1e30, -1e6])
@pytest.mark.parametrize("high", [2e38, 1.0])
@pytest.mark.parametrize("first", [16, 40, 64, 200])
def test_scores_far_above_all_before(device, fmt, dim, low, high, first):
    """Keys whose scores (base 2) are near the lowest fp32 holds, or only far below, then
    others far above them: the difference leaves fp32's range, or holds no digit of the later
    scores. The later keys take the whole weight, by their own differences: scores equal at the
    top, or spread over 4 with values that grow along them."""
    n = 260
    # base-2 score per K scale of a key of codes 96 in all dimensions but one
    unit = (dim - 1) * 96 * dim ** -0.5 * 1.4426950408889634
    cache, tables = _two_groups(device, dim, fmt, n, first, (-96, 96), (-low / unit, high / unit),
                                (7.0, 1.0))
    gen = torch.Generator(device=device).manual_seed(first)
    later = [(int(tables[0, at // 16]), at % 16) for at in range(first, n)]
    pages, slots = (torch.tensor(x, device=device) for x in zip(*later))
    spread = torch.rand(len(later), generator=gen, device=device)
    if high == 1.0:
        cache.scales[pages, 0, 0, 0, slots] *= 4 * spread
    cache.scales[pages, 0, 1, 0, slots] *= 0.5 + spread
    query = torch.ones((9, 1, dim), device=device)
    for dtype in (torch.float32, torch.bfloat16):
        _check(cache, tables, [n], [9], query.to(dtype))


@pytest.mark.parametrize("fmt", ["int8", "fp8_e4m3fn"])
@pytest.mark.parametrize("power", [-10, -7, -4])
def test_small_bf16_columns(device, power, fmt):
    """A bf16 column with one element at 2^power that meets zero codes, and the others near
    2^-19: f16's own step (2^-24) would cost those 1.5 % of themselves, 9 % of the later keys'
    weight 6 nats below the first key's. Tolerance (5e-3, relative alone): the bf16 output
    (2^-9) beside f16 weights and V scales (2^-12 each)."""
    n, dim = 100, 128
    query = torch.full((9, 2, dim), 2.0 ** -19 * (1 + 2 / 128), device=device)
    query[..., 0] = 2.0 ** power
    query = query.bfloat16()
    unit = float(query[0, 0, 1]) * (dim - 1) * 2 * 96 * dim ** -0.5  # score difference per K scale
    cache, tables = _two_groups(device, dim, fmt, n, 1, (96, -96), (6 / unit, 6 / unit), (0.0, 1.0))
    _check(cache, tables, [n], [9], query, atol=0)


@pytest.mark.parametrize("nats", [10, 12, 14])
def test_mass_in_weights_below_f16s_normal_range(device, nats):
    """Thousands of keys ``nats`` below the first: each weight is subnormal in f16, and the
    sum has to count them as the numerator does. Tolerance: half of f16's step of 2^-24 on
    each weight, and its output."""
    n, dim = 6000, 128
    unit = (dim - 1) * 2 * 96 * dim ** -0.5
    cache, tables = _two_groups(device, dim, "int8", n, 1, (96, -96), (nats / unit, nats / unit),
                                (0.0, 1.0))
    query = torch.ones((9, 1, dim), device=device)
    _check(cache, tables, [n], [9], query.half(), atol=0,
           rtol=2.0 ** -25 / np.exp(-nats) + 2.0 ** -10)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("fmt", ["int8", "fp8_e4m3fn"])
@pytest.mark.parametrize("counts,priors", [([16], [700]), ([33, 2], [250, 40]), ([250], [0]),
                                           ([300, 64], [129, 1000])])
@pytest.mark.parametrize("group", [1, 4, 8])
def test_key_halves_at_head_dim_256(device, group, counts, priors, fmt, dtype):
    """Few units at head dim 256: the waves share 64 columns and take half of every key step
    each, in units that end in either half, whole and cut into key ranges, and with padding."""
    lens = [n + p for n, p in zip(counts, priors)]
    cache, tables, gen = _cache(device, lens, 256, 1, fmt, group)
    query = torch.randn((sum(counts), group, 256), generator=gen, device=device).to(dtype)
    _check(cache, tables, lens, counts, query)
    _check(cache, tables, lens, counts, query, window=45)
    mark_padding(cache, tables, lens, 0.3, seed=3)
    _check(cache, tables, lens, counts, query)


@pytest.mark.parametrize("fmt", ["int8", "fp8_e4m3fn", "fp8_e5m2"])
@pytest.mark.parametrize("lens,counts", [([300, 90], [70, 33]), ([3000], [20])])
def test_exponents_of_padded_blocks(device, lens, counts, fmt):
    """Blocks whose V scales need exponents of 1 to 5 hold padding keys alone: they change the
    unit of the accumulators (four of them within one key step, in one piece of a split unit),
    and the result is the other blocks', of ordinary size and tolerance."""
    cache, tables, gen = _cache(device, lens, 128, 2, fmt, 17)
    large = {5: 15, 8: 18, 9: 16, 10: 17, 14: 14}  # block of a sequence: power of its scales
    for row, n in enumerate(lens):
        for block, power in large.items():
            if 16 * (block + 1) > n - counts[row]:
                continue
            cache.scales[int(tables[row, block]), :, 1] *= 2.0 ** power
            slots = int(tables[row, block]) * 16 + torch.arange(16, device=device)
            cache.write_key_valid(slots, torch.zeros(16, dtype=torch.bool, device=device))
    query = torch.randn((sum(counts), 8, 128), generator=gen, device=device)
    for dtype in (torch.float32, torch.bfloat16):
        _check(cache, tables, lens, counts, query.to(dtype))


@pytest.mark.parametrize("fmt", ["int8", "fp8_e4m3fn"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("part", [0, 256])
def test_split_units_beside_decode_rows(device, part, dtype, fmt):
    """A split chunk's partials take the workspace that the decode rows' partials, tables and
    merges of the same call used, in group 1, with padding, and with rows that see every key
    (non-causal) within a window, whose last piece takes what the bound left out."""
    counts, priors = [1, 40, 1, 1, 9], [2500, 3000, 17, 4096, 1500]
    lens = [n + p for n, p in zip(counts, priors)]
    cache, tables, gen = _cache(device, lens, 128, 2, fmt, 19)
    query = torch.randn((sum(counts), 2, 128), generator=gen, device=device).to(dtype)
    _check(cache, tables, lens, counts, query, partition_tokens=part)
    _check(cache, tables, lens, counts, query, partition_tokens=part, window=700, causal=False)
    mark_padding(cache, tables, lens, 0.2, seed=3)
    _check(cache, tables, lens, counts, query, partition_tokens=part)


def test_split_units_of_many_rows(device):
    """More chunk rows than the dispatch plan orders (256), with histories that split."""
    rng = np.random.default_rng(23)
    priors = rng.integers(0, 60, 300)
    priors[::50] = rng.integers(900, 1500, 6)
    counts = [2] * 299 + [3]
    lens = [int(n + p) for n, p in zip(counts, priors)]
    cache, tables, gen = _cache(device, lens, 64, 1, "int8", 23)
    query = torch.randn((sum(counts), 1, 64), generator=gen, device=device).half()
    _check(cache, tables, lens, counts, query)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_split_units_by_number_of_pieces(device, dtype):
    """One to sixteen pieces a unit under one bound, heads in groups of 1."""
    counts, priors = [7, 130, 3, 2], [100, 1030, 5000, 17000]
    lens = [n + p for n, p in zip(counts, priors)]
    cache, tables, gen = _cache(device, lens, 128, 1, "int8", 29)
    query = torch.randn((sum(counts), 1, 128), generator=gen, device=device).to(dtype)
    _check(cache, tables, lens, counts, query)
