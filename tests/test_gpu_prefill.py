"""Causal varlen prefill (HIP MFMA) vs an fp32 torch reference.

The reference backend's prefill is vLLM FlashAttention (backend.py:560-575),
which no reference test pins (its own check is the gather bit-exactness); the
oracle for this floating-point kernel is textbook fp32 softmax attention over
the same paged workspace, causal mask aligned bottom-right.  Tolerance
2e-2 abs + 1e-2 rel (BF16 in / out, BF16 P, fp32 accumulate).  Covers GQA
groups 1/2/4/8, ragged and single-token sequences, chunked prefill (more keys
than queries), non-causal, tails of partial key tiles and pages, and a long
sequence.
"""

from __future__ import annotations

import ctypes

import numpy as np
import pytest

from tests.conftest import gpu_available

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs a GPU")]

ATOL, RTOL = 2e-2, 1e-2
D, T = 128, 128


def _case(seed, heads, group, q_lens, k_lens):
    import torch

    g = torch.Generator().manual_seed(seed)
    q_lens = np.asarray(q_lens)
    k_lens = np.asarray(k_lens)
    B = q_lens.size
    pages = [(int(n) + T - 1) // T for n in k_lens]
    n_pages = sum(pages) + 3
    perm = torch.randperm(n_pages, generator=g).numpy()
    width = max(1, max(pages))
    bt = np.zeros((B, width), np.int32)
    used = 0
    for b, p in enumerate(pages):
        bt[b, :p] = perm[used : used + p]
        used += p
    wk = torch.randn(n_pages, T, heads, D, generator=g).to(torch.bfloat16)
    wv = torch.randn(n_pages, T, heads, D, generator=g).to(torch.bfloat16)
    nq = int(q_lens.sum())
    q = torch.randn(nq, heads * group, D, generator=g).to(torch.bfloat16)
    cu = np.concatenate([[0], np.cumsum(q_lens)]).astype(np.int32)
    return q, wk, wv, bt, cu, k_lens.astype(np.int32)


def _reference(q, wk, wv, bt, cu, k_lens, group, scale, causal):
    import torch

    out = torch.zeros(q.shape, dtype=torch.float32)
    for b in range(k_lens.size):
        q0, q1 = int(cu[b]), int(cu[b + 1])
        kl = int(k_lens[b])
        if q1 == q0:
            continue
        rows = [int(bt[b, j // T]) for j in range(kl)]
        k = wk[rows, [j % T for j in range(kl)]].float()  # [kl, H, D]
        v = wv[rows, [j % T for j in range(kl)]].float()
        qs = q[q0:q1].float()  # [ql, Hq, D]
        ql = q1 - q0
        kh = k.repeat_interleave(group, dim=1)
        vh = v.repeat_interleave(group, dim=1)
        s = torch.einsum("qhd,khd->hqk", qs, kh) * scale
        if causal:
            qi = torch.arange(ql)[:, None]
            kj = torch.arange(kl)[None, :]
            s = s.masked_fill(kj > qi + (kl - ql), float("-inf"))
        p = torch.softmax(s, dim=-1)
        out[q0:q1] = torch.einsum("hqk,khd->qhd", p, vh)
    return out


def _run(seed, heads, group, q_lens, k_lens, causal=True):
    import torch

    from fragpack_amd.ops.prefill_attn import flash_attn_varlen_func

    q, wk, wv, bt, cu, kl = _case(seed, heads, group, q_lens, k_lens)
    scale = D ** -0.5
    dev = torch.device("cuda")
    out = torch.full_like(q, float("nan"), device=dev)
    print("prefill case", seed, heads, group, list(q_lens), list(k_lens), causal, flush=True)
    flash_attn_varlen_func(q=q.to(dev), k=wk.to(dev), v=wv.to(dev), out=out,
                           cu_seqlens_q=torch.from_numpy(cu).to(dev), max_seqlen_q=int(np.max(q_lens)),
                           seqused_k=torch.from_numpy(kl).to(dev), max_seqlen_k=int(np.max(k_lens)),
                           softmax_scale=scale, causal=causal, block_table=torch.from_numpy(bt).to(dev))
    torch.cuda.synchronize()
    ref = _reference(q, wk, wv, bt, cu, kl, group, scale, causal)
    got = out.float().cpu()
    assert torch.isfinite(got).all()
    torch.testing.assert_close(got, ref, atol=ATOL, rtol=RTOL)


@pytest.mark.parametrize("group", [1, 2, 4, 8])
def test_ragged_groups(group):
    _run(1 + group, heads=2, group=group, q_lens=[1, 37, 128, 300, 64], k_lens=[1, 37, 128, 300, 64])


def test_chunked_prefill_more_keys_than_queries():
    _run(11, heads=2, group=4, q_lens=[5, 100, 129, 1], k_lens=[700, 100, 260, 999])


def test_non_causal():
    _run(12, heads=1, group=8, q_lens=[33, 200], k_lens=[90, 200], causal=False)


def test_long_sequence():
    _run(13, heads=2, group=4, q_lens=[2048], k_lens=[2048])


def test_empty_sequences_in_batch():
    _run(14, heads=2, group=2, q_lens=[0, 17, 0, 130], k_lens=[0, 17, 40, 130])


@pytest.mark.parametrize("heads,q_lens", [(3, [300, 5]), (4, [129, 64, 257]), (8, [1, 70]), (12, [260]), (16, [33, 0, 90])])
def test_workgroup_mapping(heads, q_lens):
    # head counts that split the XCDs 1, 4 and 8 ways; tile counts that are no multiple of the share
    _run(50 + heads, heads=heads, group=2, q_lens=q_lens, k_lens=[n + 40 * (i % 2) for i, n in enumerate(q_lens)])


@pytest.mark.parametrize("heads,group,q_lens,k_lens", [
    (1, 8, [70] * 5, [70] * 5),
    (3, 2, [257] * 3, [257] * 3),
    (4, 4, [130] * 2, [130, 190]),
    (6, 1, [513] * 4, [513, 600, 513, 520]),
])
def test_equal_sequences_take_turns(heads, group, q_lens, k_lens):
    # the grid's order where XCDs share a head (tile counts no multiple of the share)
    _run(90 + heads, heads=heads, group=group, q_lens=q_lens, k_lens=k_lens)


def test_a_grid_past_one_row_of_every_head():
    # 4 sequences bounded by 2^23 queries: 2^20 tiles a head, nearly all dead;
    # all 8 heads in one grid row would pass the 2^32 work items a launch takes
    import torch

    from fragpack_amd.ops.prefill_attn import flash_attn_varlen_func

    q, wk, wv, bt, cu, kl = (torch.from_numpy(x) if isinstance(x, np.ndarray) else x
                             for x in _case(61, 8, 8, [40, 1, 0, 33], [40, 130, 0, 33]))
    out = torch.full_like(q, float("nan"), device="cuda")
    print("prefill with 2^20 tiles a head", flush=True)
    flash_attn_varlen_func(q=q.cuda(), k=wk.cuda(), v=wv.cuda(), out=out, cu_seqlens_q=cu.cuda(), max_seqlen_q=1 << 23,
                           seqused_k=kl.cuda(), max_seqlen_k=130, block_table=bt.cuda())
    ref = _reference(q, wk, wv, bt.numpy(), cu.numpy(), kl.numpy(), 8, D ** -0.5, True)
    torch.testing.assert_close(out.float().cpu(), ref, atol=ATOL, rtol=RTOL)


# Grids with fewer query tiles than CUs split their keys over the CUs
# (fp_prefill_attention_split): P rounds as in the unsplit launch and only the
# order of fp32 sums differs, so a BF16 output moves by at most one step
# (2^-7 of its value), plus the sums' own rounding where terms cancel
# (2^-24 x ~100 terms' growth, of the largest |V| ~ 5: < 1e-4).
SPLITS = [
    # heads, group, q lengths, key lengths, causal
    (4, 8, [200], [8392], True),  # a short last chunk: each query tile in many parts
    (1, 1, [1], [1600], True),  # one row, one head
    (3, 2, [129, 0, 128, 1], [1700, 0, 3000, 1537], True),  # odd heads, an empty sequence, tile edges
    (8, 4, [700], [2000], True),  # ranges that end one tile and start the next
    (2, 4, [65, 64, 63], [1601, 1600, 1599], False),  # full attention
    (1, 8, [33] * 9, [1536 + 31 * i for i in range(9)], True),  # several sequences, 32-token tiles
    (2, 1, [256, 257], [1000, 1800], True),
    (1, 4, [70], [64], True),  # fewer keys than queries: rows without keys
]


@pytest.mark.parametrize("heads,group,q_lens,k_lens,causal", SPLITS)
def test_split_matches_unsplit(heads, group, q_lens, k_lens, causal):
    _split_and_unsplit(heads, group, q_lens, k_lens, causal, reference=max(k_lens) > 64)


@pytest.mark.parametrize("heads,group,q_lens,k_lens", [
    (1, 8, [1024], [34000]),  # ranges of more than 64 key tiles (flags kept 64 a time)
    (1, 1, [1 + i % 3 for i in range(70)], [1600 - 9 * i for i in range(70)]),  # more than 64 sequences
    (1, 8, [2112], [6000]),  # more than 64 query tiles of a sequence
])
def test_split_over_more_than_a_wave_of_everything(heads, group, q_lens, k_lens):
    # (the unsplit launch is the reference: checked against fp32 above)
    _split_and_unsplit(heads, group, q_lens, k_lens, True, reference=False)


def _split_and_unsplit(heads, group, q_lens, k_lens, causal, reference):
    import torch

    from fragpack_amd.ops.fragpack_ext import extension

    lib = extension()._lib
    # (a key bound that makes the split's rule hold also for short keys)
    max_q, max_k = max(q_lens), max(max(k_lens), 8192)
    q, wk, wv, bt, cu, kl = (torch.from_numpy(x) if isinstance(x, np.ndarray) else x
                             for x in _case(31 + len(q_lens), heads, group, q_lens, k_lens))
    # rows concentrated on a late key: the softmax reference moves in mid-sequence
    for b in range(len(k_lens)):
        if k_lens[b] > 1000:
            j = k_lens[b] * 2 // 3
            wk[int(bt[b, j // T]), j % T] *= 12
    width = -(-max_k // T)
    bt = torch.nn.functional.pad(bt, (0, max(0, width - bt.shape[1])))
    q, wk, wv, bt, cu, kl = (x.cuda() for x in (q, wk, wv, bt, cu, kl))
    need = lib.fp_prefill_workspace_bytes(heads, group, len(q_lens), q.shape[0], max_q, max_k)
    assert need > 0
    ws = torch.randint(0, 255, (need,), dtype=torch.uint8, device="cuda")
    outs = []
    for split in (False, True):
        print("split prefill", heads, group, q_lens, k_lens, causal, split, flush=True)
        out = torch.full_like(q, float("nan"))
        args = (q.data_ptr(), q.stride(0), wk.data_ptr(), wv.data_ptr(), wk.shape[0], heads, group, cu.data_ptr(),
                kl.data_ptr(), bt.data_ptr(), bt.stride(0), len(q_lens))
        tail = (max_q, max_k, D ** -0.5, int(causal), out.data_ptr(), out.stride(0))
        stream = torch.cuda.current_stream().cuda_stream
        if split:
            rc = lib.fp_prefill_attention_split(*args, q.shape[0], *tail, ws.data_ptr(), need, stream)
        else:
            rc = lib.fp_prefill_attention(*args, *tail, stream)
        assert rc == 0, lib.fp_last_error()
        torch.cuda.synchronize()
        outs.append(out.float())
    assert torch.isfinite(outs[0]).all()
    torch.testing.assert_close(outs[1], outs[0], atol=1e-4, rtol=2 ** -7)
    if reference:
        ref = _reference(q.cpu(), wk.cpu(), wv.cpu(), bt.cpu().numpy(), cu.cpu().numpy(), kl.cpu().numpy(), group,
                         D ** -0.5, causal)
        torch.testing.assert_close(outs[1].cpu(), ref, atol=ATOL, rtol=RTOL)


def test_split_workspace_from_the_caller_or_none_at_all(monkeypatch):
    """The caller's workspace is used in place of one from the allocator (same
    bits, no allocation); a device too full for one runs the launch that needs
    none."""
    import torch

    from fragpack_amd.ops.fragpack_ext import extension
    from fragpack_amd.ops.prefill_attn import flash_attn_varlen_func

    ext = extension()
    q, wk, wv, bt, cu, kl = (torch.from_numpy(x).cuda() if isinstance(x, np.ndarray) else x.cuda()
                             for x in _case(81, 2, 4, [120, 1], [4000, 2500]))
    assert ext._lib.fp_prefill_workspace_bytes(2, 4, 2, 121, 120, 4000) > 0

    def run(out, workspace=None):
        if workspace is None:
            return flash_attn_varlen_func(q=q, k=wk, v=wv, out=out, cu_seqlens_q=cu, max_seqlen_q=120, seqused_k=kl,
                                          max_seqlen_k=4000, block_table=bt)
        ext.prefill_attention(q, wk, wv, out, cu, kl, bt, 120, 4000, D ** -0.5, True, workspace)
        return out

    want = run(torch.empty_like(q))
    ws = torch.empty(ext.prefill_workspace_bytes(4000), dtype=torch.uint8, device="cuda")
    got, small, plain = (torch.full_like(q, float("nan")) for _ in range(3))
    whole = torch.full_like(q, float("nan"))
    empty = torch.empty
    monkeypatch.setattr(torch, "empty", lambda *a, **k: pytest.fail("allocated in the call"))
    run(got, ws)
    assert torch.equal(got, want)

    def full(*a, **k):
        raise torch.OutOfMemoryError("no memory")

    monkeypatch.setattr(torch, "empty", full)
    run(small, ws[: ws.numel() // 64])  # too small: as without one
    run(plain)
    monkeypatch.setattr(torch, "empty", empty)
    rc = ext._lib.fp_prefill_attention(q.data_ptr(), q.stride(0), wk.data_ptr(), wv.data_ptr(), wk.shape[0], 2, 4,
                                       cu.data_ptr(), kl.data_ptr(), bt.data_ptr(), bt.stride(0), 2, 120, 4000,
                                       D ** -0.5, 1, whole.data_ptr(), whole.stride(0),
                                       torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    assert torch.equal(plain, whole) and torch.equal(small, whole)


@pytest.mark.parametrize("heads,group,q_lens,k_lens", [
    (2, 1, [100, 300], [100, 500]),  # shares of a query tile are token ranges
    (3, 2, [129, 1, 128], [300, 70, 128]),
    (2, 8, [70, 33], [70, 200]),  # shares are head ranges
])
def test_four_and_eight_wave_workgroups_agree(heads, group, q_lens, k_lens):
    # the same rows per wave, so the same bits
    import torch

    runs = [_with_bounds(heads, group, q_lens, k_lens, waves, seed=71 + group)[0] for waves in (4, 8)]
    assert torch.equal(*runs)


@pytest.mark.parametrize("heads,group,q_lens,k_lens,causal", [
    (3, 1, [300, 1, 257], [700, 1, 1025], True),
    (2, 2, [129, 64], [129, 900], False),
    (1, 4, [65, 0, 200], [400, 30, 200], True),
    (5, 8, [33, 70], [97, 640], True),
    (4, 1, [256], [300], False),
])
def test_eight_wave_workgroups(heads, group, q_lens, k_lens, causal):
    got, (q, wk, wv, bt, cu, kl) = _with_bounds(heads, group, q_lens, k_lens, 8, causal)
    ref = _reference(q, wk, wv, bt, cu, kl, group, D ** -0.5, causal)
    assert got.isfinite().all()
    import torch

    torch.testing.assert_close(got.float().cpu(), ref, atol=ATOL, rtol=RTOL)


def _with_bounds(heads, group, q_lens, k_lens, waves, causal=True, seed=77):
    """The case under size bounds for which the launch runs ``waves``-wave
    workgroups: its own, or many query tiles that are not fresh prompts'
    (dead tiles leave at once)."""
    import torch

    from fragpack_amd.ops.fragpack_ext import extension
    from fragpack_amd.ops.prefill_attn import flash_attn_varlen_func

    case = q, wk, wv, bt, cu, kl = _case(seed, heads, group, q_lens, k_lens)
    rows = max(q.shape[0], max(q_lens)) if waves == 4 else 300 * 256
    max_q, max_k = (max(q_lens), max(k_lens)) if waves == 4 else (rows, 2 * rows)
    plan = (ctypes.c_int64 * 5)()
    assert extension()._lib.fp_prefill_plan(heads, group, len(q_lens), rows, max_q, max_k, int(causal), 0, plan) == 0
    assert plan[0] == waves and plan[1] == 0, list(plan)
    print("prefill waves", heads, group, q_lens, waves, flush=True)
    table = np.zeros((bt.shape[0], max(bt.shape[1], -(-max_k // T))), np.int32)
    table[:, : bt.shape[1]] = bt
    big = torch.zeros((rows, heads * group, D), dtype=torch.bfloat16, device="cuda")
    big[: q.shape[0]] = q.cuda()
    out = torch.full_like(big, float("nan"))
    flash_attn_varlen_func(q=big, k=wk.cuda(), v=wv.cuda(), out=out, cu_seqlens_q=torch.from_numpy(cu).cuda(),
                           max_seqlen_q=max_q, seqused_k=torch.from_numpy(kl).cuda(), max_seqlen_k=max_k,
                           softmax_scale=D ** -0.5, causal=causal, block_table=torch.from_numpy(table).cuda())
    return out[: q.shape[0]], case
