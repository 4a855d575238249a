"""Verify and decode calls of few sequences, whose keys are split over many waves: pieces of
a workgroup merged in LDS and long piece lists (split-KV kernel), and key pieces with their
merge (any-head-dim kernel), against float64."""

from __future__ import annotations

import pytest
import torch

from oracle import torch_f64

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
BF16, F16, E4M3, E5M2 = torch.bfloat16, torch.float16, torch.float8_e4m3fn, torch.float8_e5m2

CASES = [  # prefix, new tokens, heads, kv heads, dim, q dtype, kv dtype, window, hint of the longest chain
    # split-KV: one sequence (every workgroup inside one segment), two row blocks at D = 256
    ([9000], [4], 12, 2, 256, BF16, E5M2, -1, 4),
    ([9000], [4], 12, 2, 256, F16, F16, -1, 4),
    ([5000, 0, 3], [4, 1, 0], 16, 4, 256, BF16, BF16, -1, 4),
    ([7000, 40], [3, 7], 12, 2, 256, BF16, E4M3, 900, 7),
    ([9000] * 5 + [30], [4] * 6, 12, 2, 256, BF16, E5M2, -1, 4),    # past the one-block rule at D = 256
    ([9000], [4], 32, 8, 128, BF16, BF16, -1, 4),
    ([700, 9000, 12], [5, 5, 5], 40, 8, 128, F16, E4M3, -1, 5),
    ([4000], [4], 8, 1, 64, BF16, E5M2, -1, 4),
    ([3, 5, 2], [1, 2, 3], 8, 8, 128, BF16, BF16, -1, 3),          # fewer tiles than a workgroup has waves
    ([31] * 70, [2] * 70, 8, 2, 128, F16, F16, -1, 2),             # over 64 sequences: two scans
    # with a bound, key pieces at the tuned head dims (one 16-row block over fp16 or fp8): empty
    # sequences, a window, rows past the hint, and whole row blocks too many to split
    ([6000, 0, 700], [4, 2, 1], 32, 8, 128, F16, F16, -1, 4),
    ([6000, 0, 700], [4, 2, 0], 32, 8, 128, BF16, E4M3, 900, 4),
    ([5000, 30], [2, 1], 32, 8, 64, BF16, E5M2, -1, 2),
    ([4000, 900], [2, 3], 16, 4, 256, BF16, E4M3, -1, 3),
    ([4000, 900], [1, 4], 16, 4, 256, F16, F16, -1, 4),
    ([3000, 2000, 9], [9, 3, 1], 32, 8, 128, F16, F16, -1, 3),
    ([3000, 10], [40, 2], 8, 8, 64, BF16, E4M3, -1, 16),
    ([300, 1200] * 20, [4, 2] * 20, 32, 8, 128, F16, F16, -1, 4),
    # any-head-dim pieces: rows within and past the hint, empty sequences, windows
    ([6000], [4], 16, 4, 512, BF16, BF16, -1, 4),
    ([6000, 0, 70], [4, 3, 0], 16, 4, 512, F16, F16, -1, 4),
    ([3000], [9], 8, 2, 512, BF16, E4M3, -1, 2),
    ([3000, 100], [6, 2], 32, 8, 96, BF16, E5M2, 500, 6),
    ([3000], [4], 16, 4, 192, F16, F16, -1, 4),
    ([2500], [5], 6, 1, 48, BF16, BF16, -1, 5),
    ([2500], [40], 8, 2, 320, BF16, BF16, -1, 8),
]


def _case(prefix, new, heads, hkv, dim, q_dtype, kv):
    g = torch.Generator(device=DEV).manual_seed(11)
    seq = [p + n for p, n in zip(prefix, new)]
    slots = sum(seq) + 1
    perm = torch.randperm(slots - 1, generator=g, device=DEV) + 1
    table = torch.zeros(len(seq), max(seq) + 3, dtype=torch.int32, device=DEV)
    off = 0
    for b, n in enumerate(seq):
        table[b, :n] = perm[off:off + n].to(torch.int32)
        off += n
    k, v = (torch.randn(slots, hkv, dim, generator=g, device=DEV).to(kv) for _ in range(2))
    q = (3 * torch.randn(sum(new), heads, dim, generator=g, device=DEV)).to(q_dtype)
    qsl = [sum(new[:i]) for i in range(len(new) + 1)]
    return q, k, v, table, seq, qsl


def _run(case, prefix, window, hint, bound, workspace=None):
    from sglang_restomod_amd.attention.mi355x import ops

    q, k, v, table, seq, qsl = case
    i32 = dict(dtype=torch.int32, device=DEV)
    out = torch.full(q.shape, float("nan"), dtype=torch.float32, device=DEV)
    ops.paged_verify_forward(
        q, k, v, table, torch.tensor(seq, **i32), torch.tensor(qsl, **i32), torch.tensor(prefix, **i32),
        max_q_per_seq=hint, softmax_scale=q.shape[2] ** -0.5, k_scale=0.5, v_scale=2.0, sliding_window_size=window,
        out=out, page_size=1, max_seq_len_hint=bound, workspace=workspace)
    torch.cuda.synchronize()
    return out


@pytest.mark.parametrize("hinted", [True, False])
@pytest.mark.parametrize("prefix,new,heads,hkv,dim,q_dtype,kv,window,hint", CASES)
def test_verify_matches_float64(prefix, new, heads, hkv, dim, q_dtype, kv, window, hint, hinted):
    print(f"[case] verify split prefix={prefix[:4]} new={new[:4]} h={heads}/{hkv} d={dim} q={q_dtype} kv={kv} "
          f"window={window} hint={hint} hinted={hinted}", flush=True)
    case = _case(prefix, new, heads, hkv, dim, q_dtype, kv)
    q, k, v, table, seq, qsl = case
    out = _run(case, prefix, window, hint, max(seq) if hinted else None)
    ref = torch_f64.attend(q, k.float(), v.float(), [table[b] for b in range(len(seq))], qsl, prefix, seq,
                           softmax_scale=dim ** -0.5, k_scale=0.5, v_scale=2.0, sliding_window=window)
    # 2e-3 is the repository's bound for v_scale near 1
    assert float((out.double() - ref).abs().max()) < 4e-3


@pytest.mark.parametrize("heads,hkv,tokens,prefix", [(12, 2, 4, [190] * 16), (16, 4, 8, [300] * 20), (12, 2, 4, [9000])])
def test_fp8_d256_without_a_bound_runs_one_block_groups(heads, hkv, tokens, prefix):
    """The row groups decide how the work is shared out, so the same groups give the same
    bits: a call without a bound, and one whose bound is below four tiles per wave."""
    print(f"[case] verify d=256 without a bound h={heads}/{hkv} tokens={tokens} prefix={prefix[:2]}", flush=True)
    case = _case(prefix, [tokens] * len(prefix), heads, hkv, 256, BF16, E4M3)
    got = _run(case, prefix, -1, tokens, None)
    assert torch.equal(got, _run(case, prefix, -1, tokens, prefix[0] + tokens))
    # a bound far past the lengths takes two blocks, which sum in another order
    assert not torch.equal(got, _run(case, prefix, -1, tokens, 300_000))


@pytest.mark.parametrize("prefix,new,dim,kv", [
    ([4000] + [100] * 15, 2, 128, E4M3), ([2000] + [50] * 31, 4, 128, F16), ([2000] + [50] * 31, 2, 64, E5M2),
])
def test_a_long_sequence_among_many_short_ones_is_shared(prefix, new, dim, kv):
    """Row blocks too many to split, over a bound that one workgroup would walk for longer
    than the persistent kernel takes: the persistent kernel, as without a bound (same bits)."""
    print(f"[case] verify of {len(prefix)} ragged sequences new={new} d={dim} kv={kv}", flush=True)
    case = _case(prefix, [new] * len(prefix), 32, 8, dim, F16 if kv == F16 else BF16, kv)
    got = _run(case, prefix, -1, new, max(prefix) + new)
    assert torch.equal(got, _run(case, prefix, -1, new, None))


def test_a_small_verify_needs_no_workspace():
    """Through the C entry with none: whole row blocks, whatever the bound."""
    from sglang_restomod_amd.attention.mi355x import _lib, ops

    print("[case] verify without a workspace", flush=True)
    prefix = [4000] + [100] * 15
    case = _case(prefix, [2] * 16, 32, 8, 128, F16, F16)
    q, k, v, table, seq, qsl = case
    want = _run(case, prefix, -1, 2, max(seq))
    i32 = dict(dtype=torch.int32, device=DEV)
    seq_t, qsl_t, pre_t = torch.tensor(seq, **i32), torch.tensor(qsl, **i32), torch.tensor(prefix, **i32)
    out = torch.full(q.shape, float("nan"), dtype=torch.float32, device=DEV)
    row, head, ps, hkv, dim = ops.kv_layout(k, 1)
    rc = _lib.load().ma_paged_verify_bounded(
        q.data_ptr(), q.stride(0), q.stride(1), ops.q_dtype_code(q.dtype), q.shape[0], k.data_ptr(), v.data_ptr(), row,
        head, ops.kv_dtype_code(k.dtype), table.data_ptr(), table.stride(0), None, ps, seq_t.data_ptr(),
        qsl_t.data_ptr(), pre_t.data_ptr(), 16, 2, 32, hkv, dim, 1, -1, ops.splitkv_workgroups(q.device), dim ** -0.5,
        0.5, 2.0, max(seq), None, 0, out.data_ptr(), _lib.MA_DT_F32, out.stride(0), out.stride(1),
        torch.cuda.current_stream().cuda_stream)
    assert rc == 0, _lib.load().ma_last_error()
    torch.cuda.synchronize()
    # both within the bound of the float64 checks
    assert float((out - want).abs().max()) < 8e-3


@pytest.mark.parametrize("prefix,heads,hkv,dim,padded,bounded,kv", [
    ([700] * 16, 16, 4, 512, 512, True, BF16), ([600] * 16, 16, 4, 192, 256, False, BF16),
    ([700] * 4, 32, 8, 96, 128, True, E4M3), ([700] * 4, 32, 8, 128, 128, True, F16),
    ([700] * 16, 16, 4, 256, 256, True, E5M2), ([700] * 8, 32, 8, 64, 64, True, E4M3),
])
def test_verify_pieces_cover_the_chip_once(prefix, heads, hkv, dim, padded, bounded, kv):
    """One piece per CU at most, counted in the partial slots the call writes."""
    from sglang_restomod_amd.attention.mi355x import ops

    print(f"[case] verify pieces {len(prefix)} x {prefix[0]} h={heads}/{hkv} d={dim}", flush=True)
    case = _case(prefix, [2] * len(prefix), heads, hkv, dim, F16 if kv == F16 else BF16, kv)
    ws = ops.splitkv_workspace(torch.device(DEV), head_dim=dim).fill_(0xA5)
    _run(case, prefix, -1, 2, prefix[0] + 2 if bounded else None, ws)
    # twice as many slots as CUs, from the workspace's start (the tuned dims' workspace holds more)
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    slots = 2 * cus
    used = (ws[:slots * 16 * padded * 4].view(slots, -1) != 0xA5).any(1)
    assert len(prefix) * hkv < int(used.sum()) <= cus


@pytest.mark.parametrize("heads,hkv,dim,kv", [(8, 1, 128, BF16), (12, 2, 256, E4M3), (16, 4, 512, F16), (5, 1, 80, BF16)])
def test_decode_of_one_long_sequence(heads, hkv, dim, kv):
    """Hundreds of key pieces of one row block: more than one round of the merge's loads."""
    from sglang_restomod_amd.attention.mi355x import ops

    print(f"[case] decode pieces h={heads}/{hkv} d={dim} kv={kv}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(5)
    n = 33001
    table = (torch.randperm(n, generator=g, device=DEV) + 1).to(torch.int32).view(1, n)
    k, v = (torch.randn(n + 1, hkv, dim, generator=g, device=DEV).to(kv) for _ in range(2))
    q = (3 * torch.randn(1, heads, dim, generator=g, device=DEV)).to(F16 if kv == F16 else BF16)
    out = torch.empty(q.shape, dtype=torch.float32, device=DEV)
    ops.grouped_decode_forward(q, k, v, table, torch.tensor([n], dtype=torch.int32, device=DEV),
                               softmax_scale=dim ** -0.5, out=out, max_seq_len_hint=n, page_size=1)
    torch.cuda.synchronize()
    ref = torch_f64.attend(q, k.float(), v.float(), [table[0]], [0, 1], [n - 1], [n], softmax_scale=dim ** -0.5)
    assert float((out.double() - ref).abs().max()) < 2e-3
