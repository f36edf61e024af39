"""The stream-K merge of rows cut into many pieces (few sequences on the whole GPU) against
the float64 oracle: one piece, one round of one wave, a round of every wave, several
rounds, and rows of very different lengths in one call."""

import numpy as np
import pytest
import torch

from aster_amd import KVQuantization, PagedKVCache
from tests.gpu_util import oracle_decode

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,kv,group", [(128, 8, 4), (128, 2, 16), (64, 8, 1), (64, 4, 2),
                                          (256, 4, 8)])
@pytest.mark.parametrize("lengths", [(1,), (16,), (17,), (250,), (2049,), (6000,), (8192, 3),
                                     (4096, 0, 700, 4097, 33)])
def test_rows_of_many_pieces(device, dim, kv, group, lengths):
    gen = torch.Generator(device=device).manual_seed(sum(lengths) + dim)
    lens = np.array(lengths, np.int32)
    pages = [-(-n // 16) for n in lengths]
    perm = np.random.default_rng(dim).permutation(sum(pages) + 3).astype(np.int32)
    tables = np.zeros((len(lengths), max(pages) + 1), np.int32)
    at = 0
    for row, n in enumerate(pages):
        tables[row, :n] = perm[at:at + n]
        at += n
    cache = PagedKVCache(num_blocks=len(perm), num_layers=1, num_kv_heads=kv, head_dim=dim,
                         device=device, quantization=KVQuantization("int8"))
    cache.codes.copy_(torch.randint(-127, 128, cache.codes.shape, generator=gen, device=device,
                                    dtype=torch.int8))
    cache.scales.copy_(0.005 + 0.02 * torch.rand(cache.scales.shape, generator=gen, device=device))
    query = torch.randn((len(lengths), kv * group, dim), generator=gen, device=device).half()
    out = cache.paged_attention(0, query, torch.from_numpy(tables).to(device),
                                torch.from_numpy(lens).to(device),
                                max_context_len=max(lengths), check=True)
    want = oracle_decode(tables, cache, query, context_lens=lens, scale=dim ** -0.5, fp64=True)
    # f16 output rounding (2^-11) and f16 weights (2^-11 each, averaged over the row's keys)
    np.testing.assert_allclose(out.float().cpu().numpy(), want, atol=2e-3, rtol=2e-3)
