"""Case builders shared by the CPU and GPU test modules.

`build_paged` lays random per-sequence K/V into a cache at scattered physical
blocks (the reference's `build`, tests/test_paged_attention.py:39-65) and
`make_md` builds metadata with int32 tables (test_paged_attention.py:68-94);
both also take an index dtype so the engine's int64 contract is covered.
`int4_kernel` and `prefill_columns` ask the library which kernel a call takes.
"""

from __future__ import annotations

import ctypes
import itertools

import torch

from nanoserve_amd import _lib
from nanoserve_amd.attention import AttentionMetadata


def build_paged(seqs, num_blocks, block_size, num_kv_heads, head_dim, dtype=torch.float32,
                seed=1234, shuffle=True, fill=0.0):
    """Return (k_cache, v_cache, tables, truth) on the CPU.

    truth[i] = (K_i, V_i), each [seq_len_i, Hkv, D] in `dtype`.  Slots no
    sequence owns hold `fill`.
    """
    g = torch.Generator().manual_seed(seed)
    gp = torch.Generator().manual_seed(seed + 1)  # placement drawn apart from values
    shape = (num_blocks, block_size, num_kv_heads, head_dim)
    kc = torch.full(shape, fill, dtype=dtype)
    vc = torch.full(shape, fill, dtype=dtype)
    kf = kc.view(num_blocks * block_size, num_kv_heads, head_dim)
    vf = vc.view(num_blocks * block_size, num_kv_heads, head_dim)
    perm = torch.randperm(num_blocks, generator=gp).tolist() if shuffle else list(range(num_blocks))
    cur = 0
    tables, truth = [], []
    for sl in seqs:
        nb = -(-sl // block_size)
        table = perm[cur:cur + nb]
        cur += nb
        K = torch.randn(sl, num_kv_heads, head_dim, generator=g).to(dtype)
        V = torch.randn(sl, num_kv_heads, head_dim, generator=g).to(dtype)
        slots = torch.tensor([table[p // block_size] * block_size + p % block_size for p in range(sl)],
                             dtype=torch.long)
        if sl:
            kf.index_copy_(0, slots, K)
            vf.index_copy_(0, slots, V)
        tables.append(table)
        truth.append((K, V))
    return kc, vc, tables, truth


def make_md(seqs, query_lens, tables, block_size, device="cpu", index_dtype=torch.int32,
            with_cpu_lists=True):
    qsl = [0]
    for q in query_lens:
        qsl.append(qsl[-1] + q)
    max_seq = max(seqs)
    max_blk = max(1, -(-max_seq // block_size))
    bt = torch.zeros(len(seqs), max_blk, dtype=index_dtype)
    for i, t in enumerate(tables):
        n = min(len(t), max_blk)
        if n:
            bt[i, :n] = torch.tensor(t[:n], dtype=index_dtype)
    return AttentionMetadata(
        slot_mapping=torch.zeros(sum(query_lens), dtype=torch.long, device=device),
        query_start_loc=torch.tensor(qsl, dtype=index_dtype, device=device),
        seq_lens=torch.tensor(seqs, dtype=index_dtype, device=device),
        block_tables=bt.to(device),
        max_query_len=max(query_lens),
        max_seq_len=max_seq,
        num_seqs=len(seqs),
        num_tokens=sum(query_lens),
        is_decode_only=all(q == 1 for q in query_lens),
        query_lens_cpu=list(query_lens) if with_cpu_lists else None,
        seq_lens_cpu=list(seqs) if with_cpu_lists else None,
        query_start_loc_cpu=qsl if with_cpu_lists else None,
    )


def md_to(md: AttentionMetadata, device) -> AttentionMetadata:
    """Same metadata with every tensor moved to `device`."""
    return AttentionMetadata(
        slot_mapping=md.slot_mapping.to(device),
        query_start_loc=md.query_start_loc.to(device),
        seq_lens=md.seq_lens.to(device),
        block_tables=md.block_tables.to(device),
        max_query_len=md.max_query_len,
        max_seq_len=md.max_seq_len,
        num_seqs=md.num_seqs,
        num_tokens=md.num_tokens,
        is_decode_only=md.is_decode_only,
        query_lens_cpu=md.query_lens_cpu,
        seq_lens_cpu=md.seq_lens_cpu,
        query_start_loc_cpu=md.query_start_loc_cpu,
    )


def prefill_columns(seqs, heads):
    """Columns per prefill workgroup of a batch with these (context, new rows) sequences;
    heads is (query heads, KV heads, head size)."""
    lens = [c + q for c, q in seqs]
    qsl = [0, *itertools.accumulate(q for _, q in seqs)]
    return _lib.load().ns_paged_prefill_columns(
        (ctypes.c_int64 * len(lens))(*lens), 1, (ctypes.c_int64 * len(qsl))(*qsl), 1, len(lens), *heads)


def int4_kernel(M, N, K, gs=128, norm=False, workspace=False):
    """(kernel, tokens and features of a workgroup's tile, K splits) of an ns_int4_linear call."""
    t, f, s = ctypes.c_int32(), ctypes.c_int32(), ctypes.c_int32()
    k = _lib.load().ns_int4_linear_kernel(M, N, K, gs, norm, workspace, ctypes.byref(t), ctypes.byref(f),
                                          ctypes.byref(s))
    assert k >= 0, k
    return k, t.value, f.value, s.value


# Every (tokens, features) of a workgroup of the weight stream without a norm,
# whose waits and ring are compile-time functions of the two, with (N, K, M) that
# take it: few chunks a wave, more chunks than a scale table holds (32 and one or
# more), and split over K (a workspace given).  The last workgroup holds fewer
# tiles than the others and the last token tile is part empty.
INT4_STREAM_CASES = {
    (16, 16): ((16, 1280, 1), (16, 4224, 1), (16, 3584, 1)),
    (16, 32): ((528, 1280, 127), (528, 4224, 127), (272, 4224, 127)),
    (16, 48): ((1040, 1280, 127), (1040, 4224, 127), (544, 3584, 127)),
    (16, 64): ((2064, 1280, 100), (2064, 4224, 100), (688, 4224, 100)),
    (16, 80): ((6208, 1280, 33), (6208, 4224, 33), (3088, 3584, 33)),
    (16, 96): ((20528, 1280, 1), (20528, 4224, 1), (10928, 14336, 1)),
    (16, 112): ((24608, 1280, 1), (24608, 4224, 1), (12368, 4352, 1)),
    (16, 128): ((28688, 1280, 1), (28688, 4224, 1), (10288, 8192, 1)),
    (32, 16): ((528, 8192, 127), (528, 8192, 127), (336, 6144, 127)),
    (32, 32): ((1552, 1280, 127), (1552, 4224, 127), (528, 4224, 127)),
    (32, 48): ((2080, 1280, 127), (2080, 4224, 127), (1040, 3584, 127)),
    (32, 64): ((3088, 1280, 100), (3088, 4224, 100), (1040, 4224, 127)),
    (32, 80): ((4128, 1280, 100), (4128, 4224, 100), (1552, 3584, 127)),
    (32, 96): ((5168, 1280, 100), (5168, 4224, 100), (2576, 4864, 100)),
    (32, 112): ((6208, 1280, 100), (6208, 4224, 100), (2064, 4224, 100)),
}
