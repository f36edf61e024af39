"""Performance cases of the paged low-bit KV cache: what serving programs have it do.

A case is a dict of plain values; ``path`` names the calls it makes:

  decode     one token per sequence through ``PagedKVCache.paged_attention`` on a
             ``plan_decode`` schedule (what a decode step of several sequences runs per
             layer), with the step's K/V appended in the same call where ``append`` is set
  unplanned  the same without a schedule (callers that hold only device tables)
  step       ``append(reserved=True)`` and the varlen ``paged_attention``: prompt chunks,
             mixed steps, and the decode step of a single sequence
  append     ``append`` alone, all-or-nothing (filling a pool with finished prompts)
  engine     ``PagedAttentionRunner.forward_batch`` of a small decoder, then the rollback
             of its tokens (a draft that was not accepted)

Lengths come from the case alone, values and block tables from the seed. Histories hold
N(0, 1) keys and values quantized to the cache's format, as the benchmark's do; with
``outliers``, that share of the key rows is eight times larger.
"""

from __future__ import annotations

import math
import random
from types import SimpleNamespace

import numpy as np
import torch
from torch import nn

from aster_amd import KVQuantization, PagedAttentionRunner, PagedKVCache
from aster_amd.decode_plan import plan_decode

BLOCK = 16
DTYPES = {"float32": torch.float32, "float16": torch.float16, "bfloat16": torch.bfloat16}
FORMATS = {"int8": (torch.int8, 127.0), "fp8_e4m3fn": (torch.float8_e4m3fn, 448.0),
           "fp8_e5m2": (torch.float8_e5m2, 57344.0)}

BASE = {"path": "decode", "rows": 1, "lo": 1, "hi": 1, "mix": 0, "prefix": 0, "chunks": 0,
        "chunk_lo": 0, "chunk_hi": 0, "q_heads": 32, "kv_heads": 8, "dim": 128,
        "dtype": "bfloat16", "format": "int8", "window": 0, "padding": 0.0, "outliers": 0.0,
        "append": False}

# A decode step may attend to as many K/V bytes as the long-context case does.
MOST_KV = 16 * 32768 * 8 * 128
# ... and a step's prompt chunks to as many (query, key) pairs as the mixed step's may.
MOST_PAIRS = 8 * 512 * (4096 + 512)


def _case(name, **values):
    return {"name": name, **BASE, **values}


def listed():
    return [
        # the smallest call: four short chats of a small fp32 model, one step
        _case("tiny_decode_fp32", path="unplanned", rows=4, lo=17, hi=300, q_heads=4, kv_heads=4,
              dim=64, dtype="float32", mix=1),
        # one user alone on the card: the runner's decode step of a single sequence
        _case("single_row_step", path="step", rows=1, lo=8192, hi=8192),
        # the ordinary decode step: 64 chats of mixed lengths, the new tokens appended
        _case("batch_decode_append", rows=64, lo=128, hi=4096, append=True, mix=2),
        # a sliding-window model over an FP8 cache, long chats, fp16
        _case("window_decode_fp8", rows=48, lo=500, hi=9000, q_heads=32, kv_heads=4,
              dtype="float16", format="fp8_e4m3fn", window=1024, append=True, mix=3),
        # 256 requests behind one 2048-token system prompt
        _case("shared_prefix_decode", rows=256, lo=64, hi=512, prefix=2048, mix=4),
        # long documents: 16 contexts of 32768 tokens, 10 % large keys
        _case("long_decode", rows=16, lo=32768, hi=32768, q_heads=64, outliers=0.1, mix=5),
        # continuous batching: prompt chunks beside decoding sequences
        _case("mixed_step", path="step", rows=120, lo=256, hi=4096, chunks=8, chunk_lo=512,
              chunk_hi=512, mix=6),
        # one new prompt, no history
        _case("prompt", path="step", rows=0, lo=0, hi=0, chunks=1, chunk_lo=2000, chunk_hi=2000,
              mix=7),
        # the next chunk of one long prompt
        _case("long_prompt_chunk", path="step", rows=0, lo=16000, hi=16000, chunks=1,
              chunk_lo=512, chunk_hi=512, mix=8),
        # ragged prompts of a head-dim 64 model over an FP8 cache
        _case("ragged_prompts_fp8", path="step", rows=0, lo=0, hi=700, chunks=12, chunk_lo=33,
              chunk_hi=900, q_heads=16, kv_heads=8, dim=64, dtype="float16",
              format="fp8_e4m3fn", mix=9),
        # finished prompts written into the cache, all-or-nothing
        _case("prompt_append", path="append", rows=8, lo=512, hi=512, mix=10),
        # a whole decode step of a four-layer decoder through the runner
        _case("engine_step", path="engine", rows=16, lo=700, hi=700, q_heads=16, kv_heads=4,
              mix=11),
    ]


def _log(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.5)))))))


def draw(rng):
    path = rng.choice(["decode", "decode", "decode", "unplanned", "step", "step", "step", "step",
                       "append", "engine"])
    dim = rng.choice([64, 128, 128, 128, 256])
    kv_heads = rng.choice([2, 4, 8, 8])
    group = rng.choice([1, 2, 4, 4, 8])
    dtype = rng.choice(["bfloat16", "bfloat16", "float16", "float32"])
    case = {**BASE, "path": path, "dim": dim, "kv_heads": kv_heads, "q_heads": kv_heads * group,
            "dtype": dtype, "format": rng.choice(["int8", "int8", "int8", "fp8_e4m3fn", "fp8_e5m2"]),
            "mix": rng.randrange(1 << 20)}
    if path == "engine":
        case.update(dim=rng.choice([64, 128]), dtype=rng.choice(["bfloat16", "float16"]))
        case["lo"] = case["hi"] = _log(rng, 16, 2048)
        case["rows"] = _log(rng, 1, 48)
        return case
    if path == "append":
        case["rows"] = _log(rng, 1, 64)
        case["lo"] = _log(rng, 1, 128)
        case["hi"] = case["lo"] + rng.randrange(128)
        return case
    if rng.random() < 0.25:
        case["window"] = _log(rng, 64, 4096)
    if rng.random() < 0.15:
        case["padding"] = 0.1
    if rng.random() < 0.2:
        case["outliers"] = 0.1
    if path == "step":
        case["chunks"] = _log(rng, 1, 16)
        case["chunk_lo"] = _log(rng, 2, 1024)
        case["chunk_hi"] = min(2048, case["chunk_lo"] + rng.randrange(1, 512))
        case["rows"] = rng.choice([0, 0, _log(rng, 1, 128)])
        case["lo"] = rng.choice([0, _log(rng, 1, 8192)])
        case["hi"] = case["lo"] + _log(rng, 1, 4096)
        if dtype == "float32":
            case["rows"] = min(case["rows"], 16)
        # a drawn step's work stays at or below the mixed step's
        while _most_pairs(case) * case["q_heads"] * dim > MOST_PAIRS * 32 * 128 \
                and case["chunk_hi"] > 64:
            if case["chunks"] > 1:
                case["chunks"] //= 2
            else:
                case["chunk_hi"] //= 2
                case["chunk_lo"] = min(case["chunk_lo"], case["chunk_hi"])
        while case["rows"] * case["hi"] * kv_heads * dim > MOST_KV // 2:
            case["rows"] //= 2
        return case
    if path == "decode" and dtype == "float32":
        case["format"] = "int8"
    case["lo"] = _log(rng, 1, 8192)
    case["hi"] = case["lo"] + _log(rng, 1, 8192)
    case["rows"] = _log(rng, 2 if path == "decode" else 1, 512 if path == "decode" else 64)
    if path == "unplanned" and dtype == "float32":
        case["rows"] = min(case["rows"], 16)
    case["append"] = path == "decode" and dtype != "float32" and dim != 64 and rng.random() < 0.6
    if path == "decode" and case["window"] == 0 and rng.random() < 0.25:
        case["prefix"] = BLOCK * _log(rng, 8, 256)
        case["lo"], case["hi"] = 1 + case["lo"] % 64, 64 + case["hi"] % 512
    while case["rows"] > 2 and case["rows"] * (case["prefix"] + case["hi"]) * kv_heads * dim > MOST_KV:
        case["rows"] = case["rows"] // 2
    return case


def _most_pairs(case):
    """Upper bound of a step's (query, key) pairs over its prompt chunks."""
    return case["chunks"] * case["chunk_hi"] * (case["hi"] + case["chunk_hi"])


# ---- shapes (from the case alone) ------------------------------------------------------


def _shape(case):
    """(context lengths, query tokens) per sequence, chunk rows first. ``lo`` to ``hi`` are
    the lengths before a prompt chunk, of a decode row and of an appended prompt; a shared
    prefix comes before them."""
    rng = np.random.default_rng(case["mix"])
    prior = rng.integers(case["lo"], case["hi"], size=case["chunks"], endpoint=True)
    chunk = rng.integers(case["chunk_lo"], case["chunk_hi"], size=case["chunks"], endpoint=True)
    rows = rng.integers(max(case["lo"], 1), max(case["hi"], 1), size=case["rows"], endpoint=True)
    lens = np.concatenate([prior + chunk, rows + case["prefix"]]).astype(np.int32)
    return lens, np.concatenate([chunk, np.ones(case["rows"])]).astype(np.int32)


def _first_key(case, length, queries):
    """First key that some of a row's ``queries`` newest tokens see."""
    return max(0, length - queries - case["window"] + 1) if case["window"] else 0


def work(case):
    """K/V codes and scales of every key some query sees (a shared prefix once), queries in,
    outputs out, block ids, and the appended rows in and out; 4 q_heads dim operations per
    visible (query, key) pair."""
    item = torch.empty((), dtype=DTYPES[case["dtype"]]).element_size()
    token = case["kv_heads"] * (2 * case["dim"] + 8)
    lens, queries = _shape(case)
    if case["path"] == "append":
        rows = int(lens.sum())
        return {"bytes": rows * (token + 2 * case["kv_heads"] * case["dim"] * item + 8), "flops": 0}
    keys, pairs = 0, 0
    for length, n in zip(lens.tolist(), queries.tolist()):
        keys += length - _first_key(case, length, n)
        for part in range(0, n, 512):
            ends = np.arange(length - n + part + 1, length - n + min(n, part + 512) + 1)
            pairs += int(np.minimum(ends, case["window"]).sum() if case["window"] else ends.sum())
    if case["prefix"] and not case["window"]:
        keys -= (len(lens) - 1) * case["prefix"]
    total = int(queries.sum())
    moved = keys * token + 2 * total * case["q_heads"] * case["dim"] * item + keys // 4
    if case["append"] or case["path"] in ("step", "engine"):
        moved += total * (token + 2 * case["kv_heads"] * case["dim"] * item + 8)
    flops = 4 * case["q_heads"] * case["dim"] * pairs
    if case["path"] == "engine":
        weights = sum(p.numel() for p in _decoder(case, 0, "meta").parameters()) \
            - ENGINE["vocab"] * ENGINE["hidden"]
        return {"bytes": ENGINE["layers"] * moved + item * weights,
                "flops": ENGINE["layers"] * flops + 2 * total * weights}
    return {"bytes": moved, "flops": flops}


# ---- values ----------------------------------------------------------------------------


def _generator(seed, device="cuda"):
    return torch.Generator(device=device).manual_seed(seed)


def _quantize(x, kind):
    """The cache's quantization of rows ``[..., dim]`` in plain fp32: (codes, scales). On the
    CPU, whose division is correctly rounded, wherever a code has to be the cache's own."""
    dtype, most = FORMATS[kind]
    x = x.float()
    amax = x.abs().amax(-1)
    scales = torch.where(amax == 0, torch.ones_like(amax),
                         (amax / most).clamp_min(torch.finfo(torch.float32).tiny))
    units = (x / scales[..., None]).clamp(-most, most)
    return (units.round() if kind == "int8" else units).to(dtype), scales


def _history(case, blocks, gen):
    """Codes (as bytes) and scales of ``blocks`` full pages of random tokens."""
    shape = (2, case["kv_heads"], BLOCK, case["dim"])
    codes = torch.empty((blocks, *shape), dtype=torch.int8, device="cuda")
    scales = torch.empty((blocks, *shape[:-1]), dtype=torch.float32, device="cuda")
    for at in range(0, blocks, 2048):
        n = min(2048, blocks - at)
        x = torch.randn((n, *shape), generator=gen, device="cuda", dtype=torch.bfloat16)
        if case["outliers"]:
            large = torch.rand((n, *shape[1:-1]), generator=gen, device="cuda") < case["outliers"]
            x[:, 0] *= torch.where(large, 8.0, 1.0)[..., None].to(x.dtype)
        c, scales[at:at + n] = _quantize(x, case["format"])
        codes[at:at + n] = c.view(torch.int8)
    return codes, scales


def _tables(case, lens, seed):
    """Host block tables over a shuffled pool; a shared prefix's pages lead every row."""
    rng = np.random.default_rng([case["mix"], seed])
    lead = case["prefix"] // BLOCK
    own = [-(-int(n) // BLOCK) - lead for n in lens]
    perm = rng.permutation(lead + sum(own) + 16).astype(np.int32)
    tables = np.zeros((len(lens), lead + max(own)), dtype=np.int32)
    at = lead
    for row, n in enumerate(own):
        tables[row, :lead] = perm[:lead]
        tables[row, lead:lead + n] = perm[at:at + n]
        at += n
    return tables, len(perm)


def _inputs(case, seed):
    """Everything random of a case but the engine's: arena contents, tables and new tokens."""
    gen = _generator(seed)
    dtype = DTYPES[case["dtype"]]
    lens, queries = _shape(case)
    if case["path"] == "append":
        queries = lens
    tables, blocks = _tables(case, lens, seed)
    codes, scales = _history(case, blocks, gen)
    total = int(queries.sum())
    randn = lambda heads: torch.randn((total, heads, case["dim"]), generator=gen, device="cuda",
                                      dtype=torch.float32).to(dtype)
    query, key, value = randn(case["q_heads"]), randn(case["kv_heads"]), randn(case["kv_heads"])
    slots = np.concatenate([
        tables[row][np.arange(n - q, n) // BLOCK].astype(np.int64) * BLOCK + np.arange(n - q, n) % BLOCK
        for row, (n, q) in enumerate(zip(lens.tolist(), queries.tolist()))])
    valid = None
    if case["padding"]:
        valid = torch.rand((blocks * BLOCK,), generator=gen, device="cuda") >= case["padding"]
        valid[torch.from_numpy(slots).cuda()] = True
    return SimpleNamespace(lens=lens, queries=queries, tables=tables, blocks=blocks, codes=codes,
                           scales=scales, query=query, key=key, value=value, slots=slots,
                           valid=valid)


def prepare(case, seed):
    if case["path"] == "engine":
        return _prepare_engine(case, seed)
    x = _inputs(case, seed)
    s = SimpleNamespace(case=case, query=x.query, key=x.key, value=x.value)
    s.cache = PagedKVCache(num_blocks=x.blocks, num_layers=1, num_kv_heads=case["kv_heads"],
                           head_dim=case["dim"], device="cuda:0",
                           quantization=KVQuantization(case["format"]))
    if case["path"] != "append":  # the appends' pages are empty before
        s.cache.codes.copy_(x.codes[:, None])
        s.cache.scales.copy_(x.scales[:, None])
    if x.valid is not None:
        s.cache.write_key_valid(torch.arange(x.blocks * BLOCK, device="cuda"), x.valid)
    s.slots = torch.from_numpy(x.slots).cuda()
    s.tables, s.lens = torch.from_numpy(x.tables).cuda(), torch.from_numpy(x.lens).cuda()
    s.most = int(x.lens.max())
    s.window = case["window"] or None
    if case["path"] == "decode":
        s.plan = plan_decode(x.tables, x.lens, num_q_heads=case["q_heads"],
                             num_kv_heads=case["kv_heads"], head_dim=case["dim"],
                             q_dtype=x.query.dtype, device=s.cache.device,
                             code_format=s.cache.code_format, window=s.window)
    s.starts = torch.from_numpy(np.concatenate([[0], np.cumsum(x.queries)]).astype(np.int32)).cuda()
    s.most_queries = int(x.queries.max())
    return s


def run(s):
    path = s.case["path"]
    if path == "engine":
        return _run_engine(s)
    cache = s.cache
    if path == "append":
        cache.append(0, s.key, s.value, s.slots)
        return {"codes": cache.codes, "scales": cache.scales}
    if path == "unplanned":
        return {"out": cache.paged_attention(0, s.query, s.tables, s.lens, max_context_len=s.most,
                                             window=s.window)}
    if path == "decode":
        if not s.case["append"]:
            return {"out": cache.paged_attention(0, s.query, s.tables, s.lens,
                                                 max_context_len=s.most, window=s.window,
                                                 decode_plan=s.plan)}
        out = cache.paged_attention(0, s.query, s.tables, s.lens, max_context_len=s.most,
                                    window=s.window, decode_plan=s.plan,
                                    append=(s.key, s.value, s.slots))
    else:
        cache.append(0, s.key, s.value, s.slots, reserved=True)
        out = cache.paged_attention(0, s.query, s.tables, s.lens, max_context_len=s.most,
                                    window=s.window, query_start_loc=s.starts,
                                    max_query_len=s.most_queries)
    return {"out": out, "codes": cache.codes, "scales": cache.scales}


def tolerance(case):
    """Appends are bit-exact. Outputs: two roundings to the query's type (2^-9 relative for
    bf16, 2^-12 for fp16, at the rms 1.7e-3 and 2.1e-4), and f16 softmax weights in between
    (2e-4 to 4e-4 measured against 64 bits); four layers of a model come out at five times
    that (8e-3 measured in bf16, 1.1e-3 in fp16)."""
    if case["path"] == "append":
        return "exact"
    if case["path"] == "engine":
        return {"rel": 0.03, "max": 0.3} if case["dtype"] == "bfloat16" else {"rel": 5e-3, "max": 0.05}
    if case["dtype"] == "bfloat16":
        return {"rel": 8e-3, "max": 0.05}
    return {"rel": 2e-3, "max": 0.02}


# ---- 64-bit results --------------------------------------------------------------------


def _attend64(case, query, k, v, length, valid):
    """Outputs of the newest ``n`` tokens of one sequence: query ``[n, Hq, D]`` against the
    dequantized history ``[length, Hkv, D]``, all in 64 bits."""
    n, group = query.shape[0], case["q_heads"] // case["kv_heads"]
    out = torch.empty_like(query)
    keys = torch.arange(length, device=query.device)
    for at in range(0, n, 256):
        q = query[at:at + 256]
        pos = torch.arange(length - n + at, length - n + at + q.shape[0], device=query.device)
        seen = keys <= pos[:, None]
        if case["window"]:
            seen &= keys > pos[:, None] - case["window"]
        if valid is not None:
            seen &= valid
        for head in range(case["q_heads"]):
            kh, vh = k[:, head // group], v[:, head // group]
            scores = (q[:, head] @ kh.t().contiguous()) * case["dim"] ** -0.5
            weights = torch.softmax(scores.masked_fill(~seen, -torch.inf), -1)
            out[at:at + 256, head] = torch.nan_to_num(weights) @ vh
    return out


def exact(case, seed):
    if case["path"] == "engine":
        return _exact_engine(case, seed)
    x = _inputs(case, seed)
    slots = torch.from_numpy(x.slots).cuda()
    if case["path"] == "append":
        scales = torch.ones((x.blocks, 1, 2, case["kv_heads"], BLOCK), dtype=torch.float64,
                            device="cuda")
        for which, rows in enumerate((x.key, x.value)):
            amax = rows.double().abs().amax(-1)
            scales[slots // BLOCK, 0, which, :, slots % BLOCK] = \
                torch.where(amax == 0, 1.0, amax / FORMATS[case["format"]][1])
        return {"codes": None, "scales": scales}
    codes, scales = x.codes.view(FORMATS[case["format"]][0]), x.scales
    appends = case["append"] or case["path"] == "step"
    if appends:
        for which, rows in enumerate((x.key, x.value)):
            c, sc = _quantize(rows.cpu(), case["format"])
            x.codes[slots // BLOCK, which, :, slots % BLOCK] = c.view(torch.int8).cuda()
            scales[slots // BLOCK, which, :, slots % BLOCK] = sc.cuda()
    valid = x.valid.view(x.blocks, BLOCK) if x.valid is not None else None
    outs, at = [], 0
    for row, (length, n) in enumerate(zip(x.lens.tolist(), x.queries.tolist())):
        pages = torch.from_numpy(x.tables[row, :-(-length // BLOCK)]).cuda().long()
        kv = codes.view(torch.int8)[pages].view(codes.dtype).to(torch.float64) \
            * scales[pages][..., None].double()
        kv = kv.permute(1, 0, 3, 2, 4).reshape(2, -1, case["kv_heads"], case["dim"])[:, :length]
        real = valid[pages].reshape(-1)[:length] if valid is not None else None
        outs.append(_attend64(case, x.query[at:at + n].double(), kv[0], kv[1], length, real))
        at += n
    out = torch.cat(outs)
    return {"out": out, "codes": None, "scales": None} if appends else {"out": out}


# ---- the engine's decoder --------------------------------------------------------------

ENGINE = {"layers": 4, "hidden": 1024, "ffn": 2816, "vocab": 8192}


class _Norm(nn.Module):
    def __init__(self, width, **kw):
        super().__init__()
        self.weight = nn.Parameter(torch.ones(width, **kw))

    def forward(self, x):
        wide = x if x.dtype == torch.float64 else x.float()
        y = wide * torch.rsqrt(wide.pow(2).mean(-1, keepdim=True) + 1e-6)
        return (y * self.weight.to(wide.dtype)).to(x.dtype)


def _rope(x, positions):
    wide = torch.float64 if x.dtype == torch.float64 else torch.float32
    half = x.shape[-1] // 2
    freq = 10000.0 ** (-torch.arange(half, device=x.device, dtype=wide) / half)
    angle = positions[:, None, :, None].to(wide) * freq
    a, b = x[..., :half].to(wide), x[..., half:].to(wide)
    return torch.cat([a * angle.cos() - b * angle.sin(), a * angle.sin() + b * angle.cos()],
                     -1).to(x.dtype)


class _Attention(nn.Module):
    def __init__(self, case, **kw):
        super().__init__()
        self.num_heads, self.num_kv_heads = case["q_heads"], case["kv_heads"]
        self.head_dim, self.window, self.scale = case["dim"], None, case["dim"] ** -0.5
        width, d = ENGINE["hidden"], case["dim"]
        self.q_proj = nn.Linear(width, self.num_heads * d, bias=False, **kw)
        self.k_proj = nn.Linear(width, self.num_kv_heads * d, bias=False, **kw)
        self.v_proj = nn.Linear(width, self.num_kv_heads * d, bias=False, **kw)
        self.o_proj = nn.Linear(self.num_heads * d, width, bias=False, **kw)
        self.q_norm, self.k_norm = nn.Identity(), nn.Identity()
        self.rope = _rope


class _Mlp(nn.Module):
    def __init__(self, **kw):
        super().__init__()
        self.gate = nn.Linear(ENGINE["hidden"], ENGINE["ffn"], bias=False, **kw)
        self.up = nn.Linear(ENGINE["hidden"], ENGINE["ffn"], bias=False, **kw)
        self.down = nn.Linear(ENGINE["ffn"], ENGINE["hidden"], bias=False, **kw)

    def forward(self, x):
        return self.down(nn.functional.silu(self.gate(x)) * self.up(x))


class _Layer(nn.Module):
    def __init__(self, case, **kw):
        super().__init__()
        self.input_layernorm = _Norm(ENGINE["hidden"], **kw)
        self.self_attn = _Attention(case, **kw)
        self.post_attention_layernorm = _Norm(ENGINE["hidden"], **kw)
        self.mlp = _Mlp(**kw)


class _Decoder(nn.Module):
    def __init__(self, case, **kw):
        super().__init__()
        self.model = nn.Module()
        self.model.embed_tokens = nn.Embedding(ENGINE["vocab"], ENGINE["hidden"], **kw)
        self.model.layers = nn.ModuleList([_Layer(case, **kw) for _ in range(ENGINE["layers"])])
        self.model.norm = _Norm(ENGINE["hidden"], **kw)
        self.lm_head = nn.Linear(ENGINE["hidden"], ENGINE["vocab"], bias=False, **kw)
        self.config = SimpleNamespace(vocab_size=ENGINE["vocab"], max_position_embeddings=1 << 20)


def _decoder(case, seed, device="cuda"):
    model = _Decoder(case, device=device, dtype=DTYPES[case["dtype"]])
    if device != "meta":
        gen = _generator(seed)
        with torch.no_grad():
            for p in model.parameters():
                if p.ndim == 2:
                    p.normal_(0.0, 1.0 if p.shape[0] == ENGINE["vocab"] else p.shape[-1] ** -0.5,
                              generator=gen)
            model.lm_head.weight.mul_(ENGINE["hidden"] ** -0.5)
    return model


def _engine_inputs(case, seed):
    """Per sequence and layer the history's K/V rows, and each sequence's next token."""
    gen = _generator(seed + 1)
    shape = (case["rows"], ENGINE["layers"], 2, case["lo"], case["kv_heads"], case["dim"])
    rows = torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32)
    rng = random.Random(seed)
    return rows.to(DTYPES[case["dtype"]]), [[rng.randrange(ENGINE["vocab"])]
                                            for _ in range(case["rows"])]


def _prepare_engine(case, seed):
    rows, tokens = _engine_inputs(case, seed)
    runner = PagedAttentionRunner(
        _decoder(case, seed), policy_artifact_id="perf", backend="hip_int8_paged",
        max_blocks=case["rows"] * (case["lo"] // BLOCK + 2),
        kv_quantization=KVQuantization(case["format"]))
    runner.pool.bind_layout(num_layers=ENGINE["layers"], num_kv_heads=case["kv_heads"],
                            head_dim=case["dim"], device=torch.device("cuda", 0))
    sequences = [runner.pool.create("perf") for _ in range(case["rows"])]
    for sequence, history in zip(sequences, rows):
        runner.pool.append(sequence, tuple((layer[0], layer[1]) for layer in history))
    return SimpleNamespace(case=case, runner=runner, sequences=sequences, tokens=tokens)


def _run_engine(s):
    logits = s.runner.forward_batch(s.sequences, s.tokens)
    for sequence in s.sequences:
        s.runner.pool.truncate(sequence, s.case["lo"])
    return {"logits": torch.stack(logits)}


def _exact_engine(case, seed):
    rows, tokens = _engine_inputs(case, seed)
    model = _decoder(case, seed).double()
    kept = []
    for which in range(2):
        codes, scales = _quantize(rows[:, :, which].cpu(), case["format"])
        kept.append(codes.cuda().double() * scales.cuda()[..., None].double())
    batch, length = case["rows"], case["lo"] + 1
    positions = torch.full((batch, 1), case["lo"], device="cuda")
    with torch.inference_mode():
        hidden = model.model.embed_tokens(torch.tensor(tokens, device="cuda"))
        for index, layer in enumerate(model.model.layers):
            a, normed = layer.self_attn, layer.input_layernorm(hidden)
            split = lambda y, heads: y.view(batch, 1, heads, a.head_dim).transpose(1, 2)
            query = _rope(split(a.q_proj(normed), a.num_heads), positions)
            key = _rope(split(a.k_proj(normed), a.num_kv_heads), positions)
            value = split(a.v_proj(normed), a.num_kv_heads)
            new = []
            for y in (key, value):
                codes, scales = _quantize(y.transpose(1, 2), case["format"])
                new.append(codes.double() * scales[..., None].double())
            outs = [_attend64(case, query[b].transpose(0, 1),
                              *(torch.cat([kept[i][b, index], new[i][b]]) for i in range(2)),
                              length, None) for b in range(batch)]
            hidden = hidden + a.o_proj(torch.stack(outs).view(batch, 1, -1))
            hidden = hidden + layer.mlp(layer.post_attention_layernorm(hidden))
        logits = model.lm_head(model.model.norm(hidden))
    return {"logits": logits[:, -1].cpu()}
