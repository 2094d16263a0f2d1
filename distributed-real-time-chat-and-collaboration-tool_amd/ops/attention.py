"""Attention: varlen causal prefill and paged decode (GQA/MQA).

HIP kernels: csrc/kernels/attention_prefill.hip, csrc/kernels/attention_decode.hip.
"""
from __future__ import annotations

import math
import os

import torch

from ._ext import check, hipk, on_gpu, ptr, stream_ptr
from .gemm import Parts
from .rope import v_block_tokens

KV_BLOCK = 32  # tokens per cache block (fixed by the decode kernel)
PREFILL_QTILE = 64
# Prefill attention launch form (profiles/r2j_prefill_persistent.md): persistent
# workgroups win 9-10 % on chat-length prompts, one workgroup per (query tile,
# head group) wins on long prompts (4k tokens: 8 %); parity around 430 tokens.
PERSIST_MAX_LEN = 1024
_prefill_persist = [{"1": True, "0": False}.get(os.environ.get("DRTC_PREFILL_PERSIST", ""))]


def set_prefill_persist(on: bool | None) -> None:
    """Force the prefill attention launch form (None: per call, by the
    longest sequence of the batch)."""
    _prefill_persist[0] = None if on is None else bool(on)


def prefill_persist_for(max_len: int) -> bool:
    forced = _prefill_persist[0]
    return forced if forced is not None else max_len <= PERSIST_MAX_LEN


def prefill_form(max_len: int, ntiles: int, Hq: int, Hkv: int, D: int) -> int:
    """Launch form of the prefill attention: 1 persistent workgroups, 2 the next tile's scores ahead (four heads of 128 to a
    KV head), 0 neither.  us, plain / persistent / ahead.  A workgroup an item: persistent ones gain nothing, and ahead pays
    from 512 tokens (one prompt, 16 heads: 256 14.2 / 14.7 / 14.7, 384 17.7 / 18.2 / 17.9, 512 21.4 / 22.1 / 21.2, 700 26.4 / 27.6 /
    25.7).  More: where persistent ones lose (32 heads: 16 x 512 90 / 82 / 94, 8 x 1000 99 / 97 / 100, 8 x 1200 133.5 / 132.0 / 133.3,
    4 x 3000 324 / 334 / 317)."""
    persist = prefill_persist_for(max_len)
    G = Hq // Hkv
    if D != 128 or G % 4:
        return int(persist)
    one = ntiles * (Hq // 4) <= 256  # CUs
    if persist and (not one or _prefill_persist[0] is not None):
        return 1
    return 2 if not one or max_len >= 512 else 0


# ----------------------------------------------------------------- prefill
def prefill_tiles(cu_seqlens: list[int]) -> tuple[list[int], list[int]]:
    """Host-side 64-row query tile map for a packed batch, longest sequences
    first (causal tiles near the end of long sequences are the heaviest)."""
    seqs = []
    for s in range(len(cu_seqlens) - 1):
        n = cu_seqlens[s + 1] - cu_seqlens[s]
        for q0 in range(0, n, PREFILL_QTILE):
            seqs.append((-(q0 + PREFILL_QTILE), s, q0))
    seqs.sort()
    return [s for _, s, _ in seqs], [q for _, _, q in seqs]


def prefill_attention_ref(qkv, cu_seqlens, Hq, Hkv, D, scale, causal=True):
    T = qkv.shape[0]
    out = torch.zeros((T, Hq * D), dtype=qkv.dtype, device=qkv.device)
    G = Hq // Hkv
    cu = [int(x) for x in cu_seqlens]
    for s in range(len(cu) - 1):
        a, b = cu[s], cu[s + 1]
        if b == a:
            continue
        n = b - a
        q = qkv[a:b, : Hq * D].reshape(n, Hq, D).float().transpose(0, 1)
        k = qkv[a:b, Hq * D:(Hq + Hkv) * D].reshape(n, Hkv, D).float().transpose(0, 1)
        v = qkv[a:b, (Hq + Hkv) * D:(Hq + 2 * Hkv) * D].reshape(n, Hkv, D).float().transpose(0, 1)
        k = k.repeat_interleave(G, dim=0)
        v = v.repeat_interleave(G, dim=0)
        sc = torch.matmul(q, k.transpose(1, 2)) * scale
        if causal:
            mask = torch.ones(n, n, dtype=torch.bool, device=qkv.device).triu(1)
            sc = sc.masked_fill(mask, float("-inf"))
        o = torch.matmul(torch.softmax(sc, dim=-1), v)
        out[a:b] = o.transpose(0, 1).reshape(n, Hq * D).to(qkv.dtype)
    return out


def prefill_attention(qkv: torch.Tensor, cu_seqlens: torch.Tensor, Hq: int, Hkv: int,
                      D: int, scale: float, causal: bool = True,
                      tiles: tuple[torch.Tensor, torch.Tensor] | None = None,
                      cu_host: list[int] | None = None,
                      out: torch.Tensor | None = None,
                      max_len: int | None = None) -> torch.Tensor:
    """Packed varlen attention reading q/k/v from the fused QKV buffer.

    qkv: [T, >= (Hq + 2Hkv) * D] bf16 (RoPE already applied);
    cu_seqlens: int32 [nseq + 1]. Returns [T, Hq * D]."""
    if not on_gpu(qkv):
        return prefill_attention_ref(qkv, cu_host if cu_host is not None else cu_seqlens.tolist(),
                                     Hq, Hkv, D, scale, causal)
    assert qkv.dtype == torch.bfloat16 and qkv.stride(1) == 1
    assert qkv.shape[1] >= (Hq + 2 * Hkv) * D and Hq % Hkv == 0
    assert cu_seqlens.dtype == torch.int32 and cu_seqlens.is_cuda
    T = qkv.shape[0]
    cu = cu_host if cu_host is not None else cu_seqlens.tolist()
    if out is None:
        # rows past cu[-1] (shape padding) are not written by the kernel: zero only
        # those (zeroing the whole [T, Hq*D] output cost ~17 us per layer and chunk,
        # profiles/r2o/r2o_headline_kernel_trace.csv.gz)
        out = torch.empty((T, Hq * D), dtype=qkv.dtype, device=qkv.device)
        if cu[-1] < T:
            out[cu[-1]:].zero_()
    assert out.stride(1) == 1 and out.shape[0] == T and out.shape[1] >= Hq * D
    if tiles is None:
        assert cu[-1] <= T
        ts, tq = prefill_tiles(cu)
        dev = qkv.device
        tiles = (torch.tensor(ts, dtype=torch.int32, device=dev),
                 torch.tensor(tq, dtype=torch.int32, device=dev))
    ntiles = tiles[0].numel()
    if max_len is None:
        max_len = max((b - a for a, b in zip(cu, cu[1:])), default=0)
    check(hipk().prefill_attn(out.data_ptr(), out.stride(0), qkv.data_ptr(), qkv.stride(0),
                              Hq, Hkv, D, cu_seqlens.data_ptr(), tiles[0].data_ptr(),
                              tiles[1].data_ptr(), ntiles, float(scale), int(causal),
                              prefill_form(max_len, ntiles, Hq, Hkv, D), stream_ptr(qkv)), "prefill_attn")
    return out


# ------------------------------------------------------------------ decode
# Decode kernel variant: 1 = workgroup per (seq, kv head, partition) with a
# 4-wave LDS merge (default); 2 = one wave per (seq, kv head, partition), no
# merge.  Measured on MI355X (scripts/decode_attn_bench.py, Llama-3-8B heads):
# equal at batch 1024 (4.8 TB/s), v1 ahead at long contexts.
# 0 = pick per shape (decode_variant); 1 / 2 / 3 force a kernel variant
DECODE_VARIANT = int(os.environ.get("DRTC_DECODE_VARIANT", "0"))


def decode_variant(batch: int, Hkv: int, D: int, max_blocks: int) -> int:
    """Shape class of a decode step, named by the kernel that was the faster one for it before ``launch_variant``,
    which picks the kernel that runs; ``decode_partitioning`` cuts contexts by it (profiles/r2g_decode_persistent.md):
    3 (persistent waves, next item prefetched) when there are >= 4096
    (sequence, kv head) items and D <= 128 - the serving batches (B 1024 x 8
    kv heads: 141 vs 150 us); 2 (wave per item) when the context must be
    split over partitions to fill the chip; 1 otherwise (B 256 x ~1k tokens:
    196 vs 206 us).  Where the step's RoPE runs in the same launch
    (``fused_rope_variant``) 1 also takes the shapes of 2.
    r2l (profiles/r2l_decode_geometries.md): from 2048 items v3 also wins at
    chat lengths (Mixtral / 70B heads at B 256: 38.4 vs 40.1 / 38.9 vs 41.2 us);
    at D = 256 (Gemma-2B, one kv head) v2 wins from 1024 items (B 1024: 34.2 vs
    49.5 us; v3 holds ~400 registers there and spills).  All figures: from before kernel 1 took K through LDS."""
    if DECODE_VARIANT:
        return DECODE_VARIANT
    items = batch * Hkv
    if D <= 128 and items >= 2048:
        return 3
    if D > 128 and items >= 1024:
        return 2
    if items < 256 and max_blocks > 8:
        return 2
    return 1


def launch_variant(variant: int, max_blocks: int, max_parts: int, max_wgs: int = 0) -> int:
    """The kernel that runs where ``decode_variant`` says ``variant``: 1, since its K passes through LDS in whole rows
    and four of its workgroups fit a CU (two at heads of 256, for their LDS), where the others hold two blocks in
    registers.  us:
      32 heads of 128 over 8 kv heads, 3 / 1: 1024 x 150 tokens 139 / 115, 256 x 1000 206 / 171, 256 x 150 41 / 33, 224 x 300
        39 / 28
      32 heads of 64 over 8, 3 / 1: 256 x 150 21.6 / 20.3, 1024 x 90 52 / 48.5, 1024 x 150 76 / 69, 1024 x 500 200 / 184
      8 heads of 256 over 1, contexts of three to five quarters of the mean, rotation apart, 2 / 1: 1024 x 60 27.4 / 26.1,
        1024 x 150 44.8 / 41.5, 1024 x 400 99.8 / 80.5, 2048 x 150 82 / 72; 1024 x 20 14.6 / 15.7, and 1024 equal contexts, all of
        whose waves end together, x 150 33.7 / 37.6, x 500 102 / 91
    The table says nothing of the contexts in it: where they are of one or two blocks in a batch of 3, the kernel's waves
    take several heads to a workgroup (3 / 1: 1024 x 20 37 / 34, 1024 x 40 52 / 49, 512 x 20 21 / 20, 512 x 40 30 / 27, 256 x 40
    17 / 17; but 256 x 20 12 / 14).
    Left to the others: a choice by hand, a grid capped by ``max_wgs``, more partitions than the merge holds, and
    tables of up to three blocks, since a context of three leaves a wave without work."""
    if DECODE_VARIANT or max_wgs or max_parts > (128 if FUSED_SPLIT_MERGE else 1):
        return variant
    return variant if variant == 3 and max_blocks <= 3 else 1


# variant 1 merges split-K partitions inside the attention kernel (last
# workgroup to finish) instead of a separate decode_reduce launch
FUSED_SPLIT_MERGE = os.environ.get("DRTC_DECODE_FUSED_MERGE", "1") != "0"


def decode_partitioning(batch: int, Hkv: int, max_blocks: int, target_wgs: int = 256,
                        variant: int | None = None, D: int = 128):
    """Static (graph-capturable) split of the context into partitions.

    Returns (blocks_per_part, max_parts).  Split-K only pays when the batch
    cannot fill the chip by itself: the sweep in profiles/ shows one partition
    per sequence winning from 512 (seq, kv head) workgroups up (e.g. batch 64 x
    8 kv heads: 84 us unsplit vs 96 us in 4 parts at ~1.7k-token contexts), and
    partitions shorter than ~8 blocks losing to the merge overhead (batch 8 at
    4k tokens: 28 us with 32-block parts vs 40 us with 4-block parts)."""
    variant = variant or decode_variant(batch, Hkv, D, max_blocks)
    # a split context is some 384 workgroups, 1.5 a CU, of four waves each (launch_variant): with 1024 (one a wave)
    # 16 x 1000 tokens of 8 kv heads took 21.0 us in 5 parts, with 384 18.6 in 3; 8 x 4000 33.7 / 31.4, 1 x 16000
    # 28.9 / 25.2, 13 x 700 15.4 / 15.4
    wanted = 1.5 * target_wgs if variant == 2 else target_wgs * (4 if variant == 3 else 1)
    parts_wanted = max(1, math.ceil(wanted / max(1, batch * Hkv)))
    bpp = max(8, math.ceil(max_blocks / parts_wanted))
    bpp = ((bpp + 3) // 4) * 4
    max_parts = max(1, math.ceil(max_blocks / bpp))
    return bpp, max_parts


def paged_decode_ref(q, k_cache, v_cache, block_tables, context_lens, scale):
    B, Hq, D = q.shape
    Hkv, bs = k_cache.shape[1], k_cache.shape[2]
    G = Hq // Hkv
    out = torch.zeros((B, Hq, D), dtype=q.dtype, device=q.device)
    for b in range(B):
        ctx = int(context_lens[b])
        if ctx <= 0:
            continue
        nblk = (ctx + bs - 1) // bs
        blocks = block_tables[b, :nblk].long()
        k = k_cache[blocks].permute(1, 0, 2, 3).reshape(Hkv, nblk * bs, D)[:, :ctx].float()
        v = v_block_tokens(v_cache[blocks]).permute(1, 0, 2, 3).reshape(Hkv, nblk * bs, D)
        v = v[:, :ctx].float()
        qh = q[b].reshape(Hkv, G, D).float()
        s = torch.einsum("hgd,htd->hgt", qh, k) * scale
        p = torch.softmax(s, dim=-1)
        out[b] = torch.einsum("hgt,htd->hgd", p, v).reshape(Hq, D).to(q.dtype)
    return out


class DecodeWorkspace:
    """fp32 split-K partial buffers for one (batch bucket, partitioning)."""

    def __init__(self, batch: int, Hq: int, D: int, max_parts: int, device):
        self.max_parts = max_parts
        if max_parts > 1:
            self.part_o = torch.empty((batch, Hq, max_parts, D), dtype=torch.float32, device=device)
            self.part_ml = torch.empty((batch, Hq, max_parts, 2), dtype=torch.float32, device=device)
            # per-(sequence, kv head) arrival counters of the in-kernel split-K
            # merge (variant 1); each launch leaves them at zero
            self.counters = torch.zeros(batch * Hq, dtype=torch.int32, device=device)
        else:
            self.part_o = self.part_ml = self.counters = None


def paged_decode_attention(q: torch.Tensor, k_cache: torch.Tensor, v_cache: torch.Tensor,
                           block_tables: torch.Tensor, context_lens: torch.Tensor,
                           scale: float, out: torch.Tensor | None = None,
                           blocks_per_part: int | None = None,
                           workspace: DecodeWorkspace | None = None,
                           variant: int | None = None) -> torch.Tensor:
    """One query token per sequence against the paged cache.

    q: [B, Hq, D] view (row stride may exceed Hq*D, e.g. the fused QKV row);
    block_tables: int32 [B, max_blocks]; context_lens: int32 [B]."""
    if not on_gpu(q):
        r = paged_decode_ref(q, k_cache, v_cache, block_tables, context_lens, scale)
        if out is not None:
            out.copy_(r)
            return out
        return r
    B, Hq, D = q.shape
    assert q.dtype == torch.bfloat16 and q.stride(2) == 1 and q.stride(1) == D
    nb, Hkv, bs, D2 = k_cache.shape
    assert bs == KV_BLOCK and D2 == D and k_cache.is_contiguous() and v_cache.is_contiguous()
    assert v_cache.shape == (nb, Hkv, D, bs)
    assert Hq % Hkv == 0 and Hq // Hkv <= 16
    assert block_tables.dtype == torch.int32 and block_tables.stride(1) == 1
    assert context_lens.dtype == torch.int32 and context_lens.numel() >= B
    max_blocks = block_tables.shape[1]
    picked = variant or decode_variant(B, Hkv, D, max_blocks)
    if blocks_per_part is None or workspace is None:
        blocks_per_part, max_parts = decode_partitioning(B, Hkv, max_blocks, variant=picked, D=D)
        workspace = DecodeWorkspace(B, Hq, D, max_parts, q.device)
    variant = variant or launch_variant(picked, max_blocks, workspace.max_parts)
    if out is None:
        out = torch.empty((B, Hq, D), dtype=q.dtype, device=q.device)
    assert out.is_contiguous() and out.shape == (B, Hq, D)
    counters = ptr(workspace.counters) if variant == 1 and FUSED_SPLIT_MERGE else 0
    check(hipk().paged_decode(out.data_ptr(), ptr(workspace.part_o), ptr(workspace.part_ml),
                              counters, q.data_ptr(), q.stride(0), k_cache.data_ptr(), v_cache.data_ptr(),
                              block_tables.data_ptr(), block_tables.stride(0),
                              context_lens.data_ptr(), B, Hq, Hkv, D, float(scale),
                              workspace.max_parts, blocks_per_part, variant, stream_ptr(q)),
          "paged_decode")
    return out


# RoPE + KV write fused into the decode attention (attention_decode.hip
# DecodeRope): the step's q / k / v come unrotated from the QKV GEMM output; one launch
# per layer instead of rope_kv + attention (+ reduce).  DRTC_DECODE_FUSED_ROPE=0 keeps the launches apart.
FUSED_ROPE = os.environ.get("DRTC_DECODE_FUSED_ROPE", "1") != "0"


def fused_rope_variant(variant: int, D: int, max_parts: int, max_blocks: int = 0, max_wgs: int = 0) -> int:
    """The kernel that takes RoPE, the KV write and the merge of the partitions into the attention
    launch, or 0: 1 or 3 (``launch_variant``), a workgroup per partition of 1, so 8
    blocks are 2 per wave, and one launch instead of rope_kv, attention and decode_reduce.  Its merge
    holds up to 128 partitions.  32 heads of 128 over 8 kv heads, three launches against one:
    1 x 2000 tokens 21.9 -> 11.3 us, 1 x 16000 43.7 -> 27.0, 1 x 64000 95 -> 68, 8 x 4000 42.7 -> 31.8,
    16 x 1000 26.4 -> 19.9; two launches (one partition) against one: 40 x 1000 47.2 -> 41.8,
    64 x 300 23.2 -> 20.6, 128 x 1000 105 -> 100, 200 x 400 74.0 -> 71.5 (all before K went through LDS)."""
    if D not in (64, 128) or DECODE_VARIANT == 2:
        return 0
    variant = launch_variant(variant, max_blocks, max_parts, max_wgs)
    if variant == 3:
        return 3
    return 1 if max_parts <= (128 if FUSED_SPLIT_MERGE else 1) else 0


QKV_PARTS = 4  # attention_decode.hip kQkvParts


def decode_qkv_parts(B: int, Hkv: int, D: int, max_blocks: int, max_parts: int, max_wgs: int = 0) -> int:
    """K slices' sums that ``paged_decode_attention_rope`` adds up itself, 0 where it wants rows: its kernel 1 does, for up to
    64 rows.  us of a decode step of four layers, rows / sums: width 4096, 3 x 300 tokens 451 / 442, 8 x 500 465 / 453, 24 x
    400 510 / 498, 32 x 1000 591 / 579, 48 x 300 553 / 537, 64 x 800 646 / 629; width 2048, 20 x 500 274 / 269, 48 x 1000 329 /
    311, 64 x 300 297 / 275.  Every partition of a context reads the slices, which costs less than they give at any
    length: width 4096, 4 x 2000 463 / 458, 8 x 4000 545 / 538, 64 x 2000 830 / 819, 16 x 4000 653 / 642, 3 x 16000 597 / 592, 8 x
    12000 739 / 731; width 2048, 64 x 2000 435 / 416, 20 x 8000 494 / 491; 16 heads to a kv head, 4096 16 x 1000 486.6 /
    487.2, 16 x 4000 535.5 / 536.3, 64 x 2000 622 / 620, 3 x 16000 573 / 550, 2048 64 x 2000 349 / 335.  Beyond 64 rows the projection
    has filled the chip: 72 x 300 589 / 611, 96 x 300 621 / 640, 140 x 300 747 / 768."""
    if B > 64 or not FUSED_ROPE:
        return 0
    variant = decode_variant(B, Hkv, D, max_blocks)
    return QKV_PARTS if fused_rope_variant(variant, D, max_parts, max_blocks, max_wgs) == 1 else 0


def paged_decode_attention_rope(qkv: torch.Tensor | Parts, positions: torch.Tensor, slots: torch.Tensor,
                                cos_sin: torch.Tensor, Hq: int, Hkv: int, D: int,
                                k_cache: torch.Tensor, v_cache: torch.Tensor,
                                block_tables: torch.Tensor, context_lens: torch.Tensor,
                                scale: float, out: torch.Tensor | None = None,
                                blocks_per_part: int | None = None,
                                workspace: DecodeWorkspace | None = None,
                                max_wgs: int = 0) -> torch.Tensor:
    """Decode-step attention from the raw QKV rows [B, (Hq + 2 Hkv) D]: rotate q / k of
    the step's token (position ``positions[b]`` = context_lens[b] - 1), write its k / v
    into the paged cache at ``slots[b]`` and attend over the whole context - the result
    of ``rope_kv_`` followed by ``paged_decode_attention``.  On the GPU one launch does it at
    head sizes 64 and 128 (``fused_rope_variant``); other shapes run the two ops.
    ``max_wgs`` > 0 caps the persistent grid at that many 4-wave workgroups (attention on
    part of the chip, beside another stream's GEMMs; 0: two per CU).  ``qkv`` may be the projection's ``Parts``
    (``decode_qkv_parts``; added up ahead elsewhere)."""
    from .rope import rope_kv_

    B = qkv.shape[0]
    parts = None
    if isinstance(qkv, Parts):
        n = qkv.slab.shape[0]
        if (on_gpu(qkv.slab) and qkv.slab.dtype == torch.float32 and 2 <= n <= QKV_PARTS
                and k_cache.data_ptr() % 16 == 0 and qkv.slab.is_contiguous()
                and qkv.shape[1] % 4 == 0 and qkv.slab.data_ptr() % 16 == 0
                and blocks_per_part is not None and workspace is not None
                and n <= decode_qkv_parts(B, Hkv, D, block_tables.shape[1], workspace.max_parts, max_wgs)):
            parts = qkv
        else:
            qkv = qkv.tensor()
    fused = 1 if parts is not None else 0
    # staged into LDS: a row by whole words, K by 16-byte pieces
    if not fused and on_gpu(qkv) and FUSED_ROPE and qkv.data_ptr() % 4 == 0 and qkv.stride(0) % 2 == 0 and k_cache.data_ptr() % 16 == 0:
        variant = decode_variant(B, Hkv, D, block_tables.shape[1])
        max_parts = (workspace.max_parts if blocks_per_part is not None and workspace is not None
                     else decode_partitioning(B, Hkv, block_tables.shape[1], variant=variant, D=D)[1])
        fused = fused_rope_variant(variant, D, max_parts, block_tables.shape[1], max_wgs)
    if not fused:
        q = qkv.as_strided((B, Hq, D), (qkv.stride(0), D, 1))
        rope_kv_(qkv, positions, slots, cos_sin, Hq, Hkv, D, k_cache, v_cache, KV_BLOCK)
        return paged_decode_attention(q, k_cache, v_cache, block_tables, context_lens, scale,
                                      out=out, blocks_per_part=blocks_per_part,
                                      workspace=workspace)
    rows = qkv if parts is None else parts.slab
    assert qkv.dtype == torch.bfloat16 and rows.stride(-1) == 1
    assert qkv.shape[1] >= (Hq + 2 * Hkv) * D
    nb, hkv, bs, D2 = k_cache.shape
    assert hkv == Hkv and bs == KV_BLOCK and D2 == D and k_cache.is_contiguous()
    assert v_cache.is_contiguous() and v_cache.shape == (nb, Hkv, D, bs)
    assert positions.dtype == torch.int32 and positions.numel() >= B
    assert slots.dtype == torch.int64 and slots.numel() >= B
    assert cos_sin.dtype == torch.float32 and cos_sin.shape[1] == D and cos_sin.is_contiguous()
    assert block_tables.dtype == torch.int32 and block_tables.stride(1) == 1
    assert context_lens.dtype == torch.int32 and context_lens.numel() >= B
    if blocks_per_part is None or workspace is None:
        blocks_per_part, max_parts = decode_partitioning(B, Hkv, block_tables.shape[1],
                                                         variant=variant, D=D)
        workspace = DecodeWorkspace(B, Hq, D, max_parts, rows.device)
    if out is None:
        out = torch.empty((B, Hq, D), dtype=qkv.dtype, device=rows.device)
    assert out.is_contiguous() and out.shape == (B, Hq, D)
    # (a slab of one row is contiguous whatever that row's stride says)
    check(hipk().paged_decode_rope(out.data_ptr(), ptr(workspace.part_o), ptr(workspace.part_ml),
                                   0 if parts else rows.data_ptr(), qkv.shape[1] if parts else qkv.stride(0), k_cache.data_ptr(),
                                   v_cache.data_ptr(), block_tables.data_ptr(),
                                   block_tables.stride(0), context_lens.data_ptr(), B, Hq, Hkv, D,
                                   float(scale), workspace.max_parts, blocks_per_part,
                                   positions.data_ptr(), slots.data_ptr(), cos_sin.data_ptr(),
                                   int(max_wgs), ptr(workspace.counters), fused, stream_ptr(rows),
                                   rows.data_ptr() if parts else 0, rows.shape[0] if parts else 0), "paged_decode_rope")
    return out
