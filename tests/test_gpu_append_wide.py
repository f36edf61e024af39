"""The append's wide kernels (head dims 64 to 512) against the oracle, bit for bit, where
they can go wrong: token counts around a workgroup's tile, rows that are not 16-byte
aligned, skipped slots, scales below the fast division's range, and non-finite rows among
finite ones."""

import numpy as np
import pytest
import torch

from aster_amd import KVQuantization, PagedKVCache
from oracle import reference_cpu as ref
from tests.division_pairs import dangerous_pairs
from tests.gpu_util import arena_numpy

pytestmark = pytest.mark.gpu

HEADS = 3


def _oracle(rows, fmt):
    """Codes (bytes) and scales of ``[T, H, D]`` rows."""
    q = ref.quantize_kv_int8(rows) if fmt == "int8" else ref.quantize_kv_fp8(rows, fmt)
    return np.asarray(q.values).view(np.int8), np.asarray(q.scales)[..., 0]


@pytest.mark.parametrize("fmt", ["int8", "fp8_e4m3fn", "fp8_e5m2"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("dim", [64, 128, 256, 512])
@pytest.mark.parametrize("layout", ["packed", "strided16", "unaligned"])
def test_wide_append_bit_exact(device, dim, dtype, fmt, layout):
    tile = 2048 // dim
    for tokens in (1, tile - 1, 2 * tile + 1):
        rng = np.random.default_rng(dim + tokens)
        src = rng.standard_normal((2, tokens, HEADS, dim)).astype(np.float32)
        src[0, tokens // 2] *= 1e-4
        if dtype != torch.float16:
            src[1, -1, 0] *= 1e-25   # scale below the fast division's range
            src[0, 0, 1] = 0
        values = torch.from_numpy(src).to(dtype)
        # rows inside wider storage: the offset keeps or breaks the 16-byte alignment
        pad = {"packed": 0, "strided16": 16, "unaligned": 3}[layout]
        wide = torch.zeros((2, tokens, HEADS, dim + pad), dtype=dtype, device=device)
        rows = wide[..., pad:] if layout != "strided16" else wide[..., :dim]
        rows.copy_(values)
        blocks = (tokens + 15) // 16 + 2
        slots = rng.permutation(blocks * 16)[:tokens].astype(np.int64)
        slots[tokens // 2] = slots[tokens // 2] if tokens < 3 else -1
        cache = PagedKVCache(num_blocks=blocks, num_layers=1, num_kv_heads=HEADS, head_dim=dim,
                             device=device, quantization=KVQuantization(fmt))
        cache.append(0, rows[0], rows[1], torch.from_numpy(slots).to(device), check=True)
        got = arena_numpy(cache)
        want = [np.zeros((blocks, HEADS, 16, dim), np.int8), np.ones((blocks, HEADS, 16), np.float32)]
        for which in range(2):
            codes, scales = _oracle(values[which].float().numpy(), fmt)
            c, s = want[0].copy(), want[1].copy()
            for t in np.flatnonzero(slots >= 0):
                c[slots[t] // 16, :, slots[t] % 16] = codes[t]
                s[slots[t] // 16, :, slots[t] % 16] = scales[t]
            np.testing.assert_array_equal(got[2 * which].view(np.int8), c)
            np.testing.assert_array_equal(got[2 * which + 1], s)


@pytest.mark.parametrize("dim", [64, 256])
@pytest.mark.parametrize("bad", [np.inf, np.nan])
def test_wide_append_keeps_non_finite_rows_out(device, dim, bad):
    """Reserved slots: a non-finite row stays unwritten, a finite one is written or, where its
    workgroup saw the flag of an earlier one, left; otherwise every slot stays unwritten."""
    tokens = 2048 // dim + 3
    rng = np.random.default_rng(dim)
    key = torch.from_numpy(rng.standard_normal((tokens, HEADS, dim)).astype(np.float32)).to(torch.bfloat16)
    value = key.flip(0).clone()
    key[2, 1, dim - 1] = bad
    slots = torch.arange(tokens, dtype=torch.int64, device=device)
    for reserved in (True, False):
        cache = PagedKVCache(num_blocks=tokens // 16 + 1, num_layers=1, num_kv_heads=HEADS,
                             head_dim=dim, device=device)
        cache.append(0, key.to(device), value.to(device), slots, reserved=reserved)
        with pytest.raises(ValueError):
            cache.raise_errors()
        kc, ks, vc, vs = arena_numpy(cache)
        if not reserved:
            assert not kc.any() and not vc.any() and (ks == 1).all() and (vs == 1).all()
            continue
        codes, scales = _oracle(np.nan_to_num(key.float().numpy(), posinf=0), "int8")
        for t in range(tokens):
            for h in range(HEADS):
                if (t, h) == (2, 1):
                    assert not kc[t // 16, h, t % 16].any() and ks[t // 16, h, t % 16] == 1
                elif kc[t // 16, h, t % 16].any():
                    np.testing.assert_array_equal(kc[t // 16, h, t % 16], codes[t, h])
                    assert ks[t // 16, h, t % 16] == scales[t, h]
                else:
                    assert ks[t // 16, h, t % 16] == 1
        assert kc[2 // 16, 0, 2].any() and vc.any()  # in the flagging row's own workgroup


def _append_rows(device, rows, fmt):
    """Codes and scales of ``[T, D]`` rows through the append, as [T, D] bytes and [T]."""
    tokens, dim = rows.shape
    cache = PagedKVCache(num_blocks=-(-tokens // 16), num_layers=1, num_kv_heads=1, head_dim=dim,
                         device=device, quantization=KVQuantization(fmt))
    key = rows.to(device)[:, None]
    cache.append(0, key, key, torch.arange(tokens, device=device), check=True)
    kc, ks, vc, vs = arena_numpy(cache)
    np.testing.assert_array_equal(kc, vc)
    return kc.reshape(-1, dim)[:tokens].view(np.int8), ks.reshape(-1)[:tokens]


@pytest.mark.parametrize("fmt,offsets", [("int8", range(-1, 9)), ("fp8_e4m3fn", (-1, 0, 14, 15, 16, 17, 18)),
                                         ("fp8_e5m2", (-1, 0))])
def test_every_f16_quotient(device, fmt, offsets):
    """Row maxima of every f16 significand over elements of every f16 significand and the
    exponents at which their codes differ: up to powers of two all quotients of 16-bit input."""
    sig = torch.arange(1024, dtype=torch.int16)
    for top in range(0, 1024, 128):
        amax = (sig[top:top + 128] | (29 << 10)).view(torch.float16)
        x = torch.cat([(sig | ((28 - e) << 10)).view(torch.float16) for e in offsets])
        x = torch.cat([x, x.new_zeros(-len(x) % 511)]).reshape(-1, 511)
        x = torch.minimum(x.expand(len(amax), -1, -1), amax[:, None, None])
        rows = torch.cat([amax[:, None, None].expand(-1, x.shape[1], 1), x], 2).reshape(-1, 512)
        rows[:, 2::2] *= -1
        codes, scales = _append_rows(device, rows, fmt)
        want_codes, want_scales = _oracle(rows.float().numpy()[:, None], fmt)
        np.testing.assert_array_equal(scales, want_scales[:, 0])
        np.testing.assert_array_equal(codes, want_codes[:, 0])


@pytest.mark.parametrize("fmt,odd", [("int8", range(1, 255, 2)), ("fp8_e4m3fn", range(17, 32, 2)),
                                     ("fp8_e5m2", range(9, 16, 2))])
def test_float32_quotients_beside_ties(device, fmt, odd):
    """float32 rows whose quotients lie where the corrected product could round to the other
    side of a tie (division_pairs)."""
    most = np.float32({"int8": 127.0, "fp8_e4m3fn": 448.0, "fp8_e5m2": 57344.0}[fmt])
    rows = []
    for t, x, b in dangerous_pairs(odd):
        x, b = np.float32(x), np.float32(b)
        amax = np.float32(most * b)
        if amax / most != b:
            continue  # no row has this scale
        tie = t / 2 if fmt == "int8" else t
        x = np.ldexp(x, int(np.round(np.log2(tie * b / x))))
        row = np.zeros(64, np.float32)
        row[:3] = amax, x, -x
        rows.append(row)
    assert len(rows) > 20
    rows = np.stack(rows)
    codes, scales = _append_rows(device, torch.from_numpy(rows), fmt)
    want_codes, want_scales = _oracle(rows[:, None], fmt)
    np.testing.assert_array_equal(scales, want_scales[:, 0])
    np.testing.assert_array_equal(codes, want_codes[:, 0])
