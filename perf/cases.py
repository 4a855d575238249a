"""The attention calls whose speed this repository is measured by.

An engine makes these calls once per layer and forward: a decode step, the verification of
a linear draft, and the extend (prefill) of new prompt tokens over a cached prefix, over
16-bit and fp8 token pools. Most of the listed cases call the operators
(``grouped_decode_forward``, ``paged_forward``); the ``layer_*`` ones go through
``MI355XAttnBackend`` as the engine does: metadata of the batch, the write of the new K and V
into the pool, attention.

Values: q, k and v are standard normal, as the models' normalised and rotated heads are at
scale ``dim ** -0.5`` (scores of about unit variance); fp8 pools hold ``x / scale``. Slots are
a random permutation of the whole pool (page size 1), or pages of 16 in random order.
Sequence lengths are part of a case (drawn from its ``lens``), everything else comes from the
seed of ``prepare``.
"""

from __future__ import annotations

import random
from types import SimpleNamespace

import torch

from sglang_restomod_amd.attention.mi355x import ops
from sglang_restomod_amd.attention.mi355x.backend import MI355XAttnBackend

DEVICE = "cuda:0"
DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16,
          "e4m3": torch.float8_e4m3fn, "e5m2": torch.float8_e5m2}


def _case(mode, batch, prefix, new, heads, heads_kv, dim, dtype, kv, *, entry="op", window=-1, page=1, lens=0,
          name=None):
    """``prefix`` and ``new``: inclusive ranges of the cached and the new tokens of a sequence."""
    c = {} if name is None else {"name": name}
    c.update(mode=mode, entry=entry, batch=batch, prefix_lo=prefix[0], prefix_hi=prefix[1], new_lo=new[0],
             new_hi=new[1], heads=heads, heads_kv=heads_kv, dim=dim, dtype=dtype, kv=kv, window=window, page=page,
             lens=lens)
    return c


def listed():
    return [
        # one user, a short context: the latency of a single small call
        _case("decode", 1, (511, 511), (1, 1), 32, 8, 128, "fp16", "fp16", name="decode_single"),
        # a full decode batch of a 70B-class model's heads
        _case("decode", 64, (1023, 8191), (1, 1), 64, 8, 128, "bf16", "bf16", lens=1, name="decode_batch"),
        # long contexts, many users, an fp8 pool: the largest pool
        _case("decode", 128, (4095, 32767), (1, 1), 32, 8, 128, "bf16", "e4m3", lens=3, name="decode_fp8_long"),
        # a decode layer of an engine step with a sliding window, K/V write included
        _case("decode", 16, (511, 8191), (1, 1), 32, 8, 128, "fp16", "fp16", entry="layer", window=4096, lens=5,
              name="layer_decode_window"),
        # speculative decoding: verification of 4 draft tokens for a full batch
        _case("verify", 32, (2048, 16384), (4, 4), 64, 8, 128, "bf16", "bf16", lens=4, name="verify_batch"),
        # the same for a few users at a 27B model's two-GPU share (head dim 256), paged fp8 pool
        _case("verify", 6, (2048, 32768), (4, 4), 12, 2, 256, "bf16", "e5m2", page=16, lens=6,
              name="verify_fp8_d256"),
        # prefill of a mixed batch of prompts over cached prefixes
        _case("extend", 8, (0, 4096), (256, 2048), 40, 8, 128, "bf16", "bf16", lens=2, name="extend_batch"),
        # one chunk of a long prompt (chunked prefill far into the context)
        _case("extend", 1, (28001, 28001), (1021, 1021), 32, 8, 128, "bf16", "bf16", lens=7, name="extend_chunk"),
        # short chat turns over a cached system prompt
        _case("extend", 4, (64, 1500), (9, 130), 32, 8, 128, "fp16", "fp16", lens=8, name="extend_short"),
        # prefill at head dim 256 (a 27B model's two-GPU share)
        _case("extend", 8, (0, 4096), (256, 2048), 12, 2, 256, "bf16", "bf16", lens=2, name="extend_d256"),
        # prefill at the widest head dim
        _case("extend", 4, (0, 4096), (256, 2048), 16, 4, 512, "bf16", "bf16", lens=9, name="extend_d512"),
        # a prefill layer of an engine step over an fp8 pool, quantizing write included
        _case("extend", 8, (0, 4096), (256, 2048), 40, 8, 128, "bf16", "e4m3", entry="layer", lens=12,
              name="layer_extend_fp8"),
    ]


# (query heads, kv heads, head dim) of this repository's workloads and tests
_HEADS = [(32, 8, 128), (64, 8, 128), (40, 8, 128), (8, 1, 128), (12, 2, 256), (16, 4, 256), (16, 4, 512),
          (32, 8, 64), (32, 8, 96), (16, 4, 192)]
_KV = [("fp16", "fp16"), ("bf16", "bf16"), ("bf16", "bf16"), ("bf16", "e4m3"), ("bf16", "e5m2")]
_MAX_BYTES = 4.0e9    # below decode_fp8_long
_MAX_FLOPS = 4.5e11   # at most extend_batch's time at head dims up to 256, extend_d512's at 512


def _log(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    mode = rng.choice(["decode", "decode", "verify", "extend", "extend"])
    entry = "layer" if mode != "verify" and rng.random() < 0.25 else "op"
    heads, heads_kv, dim = rng.choice(_HEADS)
    dtype, kv = rng.choice(_KV)
    window = rng.choice([-1, -1, -1, 1024, 4096])
    page = rng.choice([1, 1, 16]) if entry == "op" else 1
    if mode == "decode":
        batch, new = _log(rng, 1, 128), (1, 1)
        lo = _log(rng, 128, 16384)
    elif mode == "verify":
        batch, n = _log(rng, 1, 32), rng.randint(2, 8)
        new = (n, n)
        lo = _log(rng, 256, 16384)
    else:
        batch = _log(rng, 1, 16)
        top = _log(rng, 16, 4096)
        new = (max(1, top // 8), top)
        lo = _log(rng, 1, 16384)
    hi = lo + rng.randint(0, lo)
    case = _case(mode, batch, (lo, hi), new, heads, heads_kv, dim, dtype, kv, entry=entry, window=window, page=page,
                 lens=rng.randint(100, 10 ** 6))
    while True:
        w = work(case)
        if w["bytes"] <= _MAX_BYTES and w["flops"] <= _MAX_FLOPS:
            return case
        if case["batch"] > 1:
            case["batch"] -= max(1, case["batch"] // 4)
        else:
            case["prefix_lo"] //= 2
            case["prefix_hi"] //= 2


def _lengths(case):
    """(prefix, new) tokens of each sequence."""
    r = random.Random(case["lens"])
    return [(r.randint(case["prefix_lo"], case["prefix_hi"]), r.randint(case["new_lo"], case["new_hi"]))
            for _ in range(case["batch"])]


def work(case):
    """The visible K and V read once, the slots (or pages) of those keys, q in and out; 4 D flop
    per visible (query row, key) pair. A layer also reads the new K and V and writes them."""
    heads, hkv, dim = case["heads"], case["heads_kv"], case["dim"]
    kvb = 1 if case["kv"] in ("e4m3", "e5m2") else 2
    w = case["window"]
    tokens = keys = pairs = 0
    for p, n in _lengths(case):
        tokens += n
        keys += p + n if w < 0 else min(p + n, w + n)
        if w < 0:
            pairs += n * p + n * (n + 1) // 2
        else:
            short = max(0, min(n, w - p))  # query i sees min(p + i, w) + 1 keys
            pairs += short * p + short * (short + 1) // 2 + (n - short) * (w + 1)
    nbytes = keys * (2 * hkv * dim * kvb) + 4 * ((keys + case["page"] - 1) // case["page"])
    nbytes += 2 * tokens * heads * dim * 2
    if case["entry"] == "layer":
        nbytes += tokens * (2 * hkv * dim * (2 + kvb) + 8)
    return {"bytes": nbytes, "flops": 4 * dim * heads * pairs}


def _inputs(case, seed):
    """Host lengths and device tensors of a case, from the seed."""
    g = torch.Generator(device=DEVICE).manual_seed(seed)
    lens = _lengths(case)
    heads, hkv, dim, page = case["heads"], case["heads_kv"], case["dim"], case["page"]
    qdt, kvdt = DTYPES[case["dtype"]], DTYPES[case["kv"]]
    seq = [p + n for p, n in lens]
    units = [(n + page - 1) // page for n in seq]  # pages of each sequence
    total = sum(units) + 1                         # page 0 is padding
    perm = (torch.randperm(total - 1, generator=g, device=DEVICE) + 1).to(torch.int32)
    rows = (torch.randperm(len(seq), generator=g, device=DEVICE) + 1).tolist()
    table = torch.zeros(len(seq) + 1, max(units) + 1, dtype=torch.int32, device=DEVICE)
    off = 0
    for r, n in zip(rows, units):
        table[r, :n] = perm[off:off + n]
        off += n
    s = SimpleNamespace(lens=lens, seq=seq, rows=rows, table=table, scale=dim ** -0.5, k_scale=1.0, v_scale=1.0)
    if kvdt.itemsize == 1:
        s.k_scale, s.v_scale = 0.5 + 1.5 * random.Random(seed).random(), 0.5 + 1.5 * random.Random(seed + 1).random()

    def pool(scale):
        x = torch.empty(total * page, hkv, dim, dtype=kvdt, device=DEVICE)
        for i in range(0, x.shape[0], 1 << 18):
            part = torch.randn(min(1 << 18, x.shape[0] - i), hkv, dim, generator=g, device=DEVICE)
            x[i:i + (1 << 18)] = (part / scale).to(kvdt) if kvdt.itemsize == 1 else part.to(kvdt)
        return x

    s.k_pool, s.v_pool = pool(s.k_scale), pool(s.v_scale)
    tokens = sum(n for _, n in lens)
    s.q = torch.randn(tokens, heads, dim, generator=g, device=DEVICE).to(qdt)
    if case["entry"] == "layer":
        s.k_new = torch.randn(tokens, hkv, dim, generator=g, device=DEVICE).to(qdt)
        s.v_new = torch.randn(tokens, hkv, dim, generator=g, device=DEVICE).to(qdt)
        s.loc = torch.cat([table[r, p:p + n] for r, (p, n) in zip(rows, lens)]).to(torch.int64)
    return s


def prepare(case, seed):
    s = _inputs(case, seed)
    s.mode, s.entry, s.window, s.page = case["mode"], case["entry"], case["window"], case["page"]
    i32 = dict(dtype=torch.int32, device=DEVICE)
    s.row_index = torch.tensor(s.rows, dtype=torch.int64, device=DEVICE)
    s.seq_lens = torch.tensor(s.seq, **i32)
    s.prefix_lens = torch.tensor([p for p, _ in s.lens], **i32)
    new = [n for _, n in s.lens]
    s.query_start_loc = torch.tensor([sum(new[:i]) for i in range(len(new) + 1)], **i32)
    s.max_len, s.max_new = max(s.seq), max(new)
    if s.page > 1:  # the paged view of the pool
        s.k_pool = s.k_pool.view(-1, s.page, *s.k_pool.shape[1:])
        s.v_pool = s.v_pool.view(-1, s.page, *s.v_pool.shape[1:])
    if s.entry == "layer":
        _engine(case, s, new)
    return s


def _engine(case, s, new):
    """The engine's objects: model runner with its token pool, layer, forward batch."""
    hkv, dim = case["heads_kv"], case["dim"]
    pool = SimpleNamespace(get_key_buffer=lambda layer_id: s.k_pool, get_value_buffer=lambda layer_id: s.v_pool)
    runner = SimpleNamespace(
        device=DEVICE, page_size=1, token_to_kv_pool=pool, kv_cache_dtype=s.k_pool.dtype,
        model_config=SimpleNamespace(context_len=int(s.table.shape[1]), head_dim=dim, v_head_dim=dim),
        req_to_token_pool=SimpleNamespace(req_to_token=s.table, size=int(s.table.shape[0])))
    fp8 = s.k_pool.dtype.itemsize == 1
    s.layer = SimpleNamespace(
        layer_id=0, tp_q_head_num=case["heads"], tp_k_head_num=hkv, tp_v_head_num=hkv, head_dim=dim, qk_head_dim=dim,
        v_head_dim=dim, scaling=s.scale, sliding_window_size=s.window, is_cross_attention=False,
        attn_type=SimpleNamespace(name="DECODER"), logit_cap=0.0, xai_temperature_len=-1,
        k_scale=torch.tensor(s.k_scale, device=DEVICE) if fp8 else None,
        v_scale=torch.tensor(s.v_scale, device=DEVICE) if fp8 else None,
        k_scale_float=s.k_scale, v_scale_float=s.v_scale)
    decode = s.mode == "decode"
    mode = SimpleNamespace(is_decode_or_idle=lambda: decode, is_extend=lambda: not decode,
                           is_target_verify=lambda: False, is_draft_extend=lambda: False,
                           is_draft_extend_v2=lambda: False)
    s.batch = SimpleNamespace(
        forward_mode=mode, batch_size=len(s.seq), req_pool_indices=s.row_index, seq_lens=s.seq_lens.to(torch.int64),
        seq_lens_cpu=torch.tensor(s.seq, dtype=torch.int64), out_cache_loc=s.loc, spec_info=None,
        extend_seq_lens=torch.tensor(new, dtype=torch.int32, device=DEVICE), extend_prefix_lens=s.prefix_lens,
        extend_seq_lens_cpu=new)
    s.backend = MI355XAttnBackend(runner)
    s.q2, s.k2, s.v2 = (x.reshape(x.shape[0], -1) for x in (s.q, s.k_new, s.v_new))


def run(s):
    if s.entry == "layer":
        s.backend.init_forward_metadata(s.batch)
        out = s.backend.forward(s.q2, s.k2, s.v2, s.layer, s.batch)
        if s.k_pool.dtype.itemsize == 1:
            return out, s.k_pool.view(torch.uint8), s.v_pool.view(torch.uint8)
        return out, s.k_pool, s.v_pool
    if s.mode == "decode":
        return ops.grouped_decode_forward(
            s.q, s.k_pool, s.v_pool, s.table, s.seq_lens, softmax_scale=s.scale, k_scale=s.k_scale,
            v_scale=s.v_scale, row_index=s.row_index, page_size=s.page, sliding_window_size=s.window,
            max_seq_len_hint=s.max_len)
    out, _ = ops.paged_forward(  # the second result is an unfilled buffer
        s.q, s.k_pool, s.v_pool, s.table, s.seq_lens, s.query_start_loc, s.prefix_lens, block_size=s.page,
        softmax_scale=s.scale, sliding_window_size=s.window, linear_verify=s.mode == "verify", k_scale=s.k_scale,
        v_scale=s.v_scale, max_seq_len_hint=s.max_len, row_index=s.row_index,
        max_q_len_hint=s.max_new if s.mode == "verify" else None)
    return out


def tolerance(case):
    """About four times what the path shows against 64 bits: 1.7e-3 and 9e-3 in bf16 (the
    output's own rounding and, in the extend, P in fp16), 4.5e-4 and 2e-3 in fp16."""
    if case["dtype"] == "bf16":
        return {"rel": 7e-3, "max": 3.6e-2}
    return {"rel": 1.8e-3, "max": 8e-3}


def exact(case, seed):
    s = _inputs(case, seed)
    heads, hkv, dim, page, window = case["heads"], case["heads_kv"], case["dim"], case["page"], case["window"]
    g = heads // hkv
    layer = case["entry"] == "layer"
    if layer:
        kvdt = s.k_pool.dtype
        fp8 = kvdt.itemsize == 1
        s.k_pool[s.loc] = (s.k_new / s.k_scale).to(kvdt) if fp8 else s.k_new
        s.v_pool[s.loc] = (s.v_new / s.v_scale).to(kvdt) if fp8 else s.v_new
    out = torch.empty(s.q.shape, dtype=torch.float64, device=DEVICE)
    t0 = 0
    for r, (p, n) in zip(s.rows, s.lens):
        pos = torch.arange(p + n, device=DEVICE)
        slots = s.table[r, pos // page].to(torch.int64) * page + pos % page
        k = s.k_pool[slots].to(torch.float64) * s.k_scale
        v = s.v_pool[slots].to(torch.float64) * s.v_scale
        qpos = p + torch.arange(n, device=DEVICE)
        hide = pos[None, :] > qpos[:, None]
        if window >= 0:
            hide |= pos[None, :] < qpos[:, None] - window
        for h in range(hkv):
            for i in range(0, n, 512):
                e = min(n, i + 512)
                q = s.q[t0 + i:t0 + e, h * g:(h + 1) * g].to(torch.float64).reshape(-1, dim)
                score = (q @ k[:, h].t().contiguous()) * s.scale
                score = score.view(e - i, g, -1).masked_fill_(hide[i:e, None, :], float("-inf"))
                prob = torch.softmax(score, dim=-1).view(q.shape[0], -1)
                out[t0 + i:t0 + e, h * g:(h + 1) * g] = (prob @ v[:, h].contiguous()).view(e - i, g, dim)
        t0 += n
    if not layer:
        return out
    return out.reshape(out.shape[0], -1), None, None
