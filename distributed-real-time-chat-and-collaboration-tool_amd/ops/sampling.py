"""Token sampling: greedy / temperature + top-k + top-p.

HIP kernel: csrc/kernels/sampling.hip (one workgroup per row; graph-replayable
because the RNG step counter lives in device memory).
"""
from __future__ import annotations

import torch

from ._ext import check, hipk, on_gpu, ptr, stream_ptr

MAX_CANDIDATES = 1024


def sample_ref(logits: torch.Tensor, temperature: torch.Tensor | None = None,
               top_k: torch.Tensor | None = None, top_p: torch.Tensor | None = None,
               generator: torch.Generator | None = None) -> torch.Tensor:
    """Reference semantics of the HIP sampler (draws differ: torch RNG).

    * temperature <= 0: argmax.
    * 0 < top_k < V: the tokens whose logit is >= the k-th largest (k capped
      at MAX_CANDIDATES; ties with the k-th value kept), softmax(l / T) over
      them, cut at the first sorted position whose inclusive mass reaches
      top_p, draw.
    * top_k == 0 (or >= V): exact top-p over the whole vocabulary: token i is
      kept iff the probability mass of tokens STRICTLY more likely than i is
      < top_p (so tied tokens are kept or dropped together)."""
    B, V = logits.shape
    out = torch.empty(B, dtype=torch.int32, device=logits.device)
    lf = logits.float()
    for b in range(B):
        t = float(temperature[b]) if temperature is not None else 0.0
        if t <= 0:
            out[b] = int(torch.argmax(lf[b]))
            continue
        pp = float(top_p[b]) if top_p is not None and 0 < float(top_p[b]) < 1 else 1.0
        k = int(top_k[b]) if top_k is not None else 0
        if 0 < k < V:
            k = min(k, MAX_CANDIDATES)
            kth = torch.topk(lf[b], k).values[-1]
            idx = torch.nonzero(lf[b] >= kth).flatten()
            vals = lf[b, idx]
            order = torch.argsort(-vals, stable=True)
            vals, idx = vals[order], idx[order]
            p = torch.softmax(vals / t, dim=-1)
            cum = torch.cumsum(p, 0)
            cut = int(torch.searchsorted(cum, torch.tensor(pp * float(cum[-1]))))
            cut = min(cut, len(idx) - 1)
            p = p[: cut + 1]
            j = int(torch.multinomial(p / p.sum(), 1, generator=generator))
            out[b] = int(idx[j])
            continue
        vals, idx = torch.sort(lf[b], descending=True, stable=True)
        p = torch.softmax(vals / t, dim=-1)
        if pp < 1.0:
            # mass strictly above each token: the exclusive cumsum at the first
            # position holding its value
            excl = torch.cumsum(p, 0) - p
            first = torch.searchsorted(-vals, -vals, right=False)
            keep = excl[first] < pp
            p = p * keep
        j = int(torch.multinomial(p / p.sum(), 1, generator=generator))
        out[b] = int(idx[j])
    return out


def sample(logits: torch.Tensor, temperature: torch.Tensor | None = None,
           top_k: torch.Tensor | None = None, top_p: torch.Tensor | None = None,
           seed: int = 0, step: torch.Tensor | None = None,
           out: torch.Tensor | None = None,
           mirror: tuple[torch.Tensor, list[torch.Tensor]] | None = None) -> torch.Tensor:
    """logits [B, V] bf16 -> int32 token ids [B].

    ``mirror``: (turn, two pinned int32 buffers), behind ``step_stage`` on the GPU: the tokens go to the buffer of the set
    that it read as well.

    temperature/top_k/top_p are per-row device tensors (float32 / int32 /
    float32); ``step`` is an int64 device scalar the caller advances.  On the GPU a
    row without a number above -inf gets -1 (``sample_ref`` raises)."""
    if not on_gpu(logits):
        # counter-based like the HIP sampler: the draws are a function of (seed, step), so a
        # step re-run with the same counter (EP capacity redo) draws the same tokens
        gen = None
        if step is not None:
            gen = torch.Generator().manual_seed(
                (seed * 0x9E3779B1 + int(step.reshape(-1)[0])) & 0x7FFFFFFFFFFFFFFF)
        r = sample_ref(logits, temperature, top_k, top_p, generator=gen)
        if out is not None:
            out.copy_(r)
            return out
        return r
    assert logits.dim() == 2 and logits.dtype == torch.bfloat16 and logits.stride(1) == 1
    B, V = logits.shape
    for t, dt in ((temperature, torch.float32), (top_k, torch.int32), (top_p, torch.float32)):
        assert t is None or (t.dtype == dt and t.numel() >= B and t.is_cuda)
    assert step is None or (step.dtype == torch.int64 and step.is_cuda)
    if out is None:
        out = torch.empty(B, dtype=torch.int32, device=logits.device)
    assert out.dtype == torch.int32 and out.is_contiguous()
    turn, hosts = mirror or (None, (None, None))
    assert turn is None or turn.dtype == torch.int32 and turn.is_cuda
    for h in hosts if mirror else ():
        assert h.dtype == torch.int32 and h.is_contiguous() and h.numel() >= B and h.is_pinned()
    check(hipk().sample(out.data_ptr(), logits.data_ptr(), B, V, logits.stride(0),
                        ptr(temperature), ptr(top_k), ptr(top_p), int(seed) & ((1 << 64) - 1),
                        ptr(step), ptr(turn), ptr(hosts[0]), ptr(hosts[1]), stream_ptr(logits)), "sample")
    return out


class StageRows:
    """``dst[a:b] = host[a:b]`` for the byte ranges (a, b), multiples of 4, of two uint8 buffers of one size, at every call.
    ``table`` (at, rows, columns, lengths, per): of the 32-bit words [rows, columns] at byte ``at`` also, row r's first
    ceil(length / per) at least, its length the r-th 32-bit word of ``host`` from byte ``lengths`` on.
    On the GPU ``host`` is pinned, and a kernel reads it: it stays unchanged until the stream is past it."""

    def __init__(self, dst: torch.Tensor, host: torch.Tensor, ranges: list[tuple[int, int]],
                 table: tuple[int, int, int, int, int] | None = None):
        assert dst.shape == host.shape and dst.dtype == host.dtype == torch.uint8
        assert dst.is_contiguous() and host.is_contiguous()
        at, rows, columns, lengths, per = table or (0, 0, 0, 0, 1)
        whole, n = (at, at + 4 * rows * columns), dst.numel()
        assert all(0 <= a <= b <= n and a % 4 == b % 4 == 0 for a, b in [*ranges, whole, (lengths, lengths + 4 * rows)])
        assert rows >= 0 and columns >= 0 and per >= 1
        self.dst, self.host, self.ranges = dst, host, [*ranges, whole]
        self.kernel = on_gpu(dst) and host.is_pinned()
        self.args = dst.data_ptr(), host.data_ptr(), [(a // 4, (b - a) // 4) for a, b in ranges]
        self.table = at // 4, rows, columns, lengths // 4, per

    def __call__(self) -> None:
        if self.kernel:
            check(hipk().stage_rows(*self.args, stream_ptr(self.dst), self.table), "stage_rows")
            return
        for a, b in self.ranges:
            self.dst[a:b].copy_(self.host[a:b])


def step_stage(stages: list[StageRows], ids: torch.Tensor, src: int, host: int, sampled: torch.Tensor,
               counter: torch.Tensor, position: torch.Tensor, turn: torch.Tensor) -> None:
    """One of two ``StageRows`` of one destination and ranges, and ``step_begin`` with src and host at these byte offsets of
    its staging set, in one launch: the set is ``turn[0]``, which the launch gives to the other one (int32 [2], [1] 0)."""
    a, b = stages
    B, size = ids.numel(), a.dst.numel()
    assert a.kernel and b.kernel and a.dst is b.dst and a.ranges == b.ranges and a.table == b.table
    assert src % 8 == host % 4 == 0 and 0 <= src <= size - 8 * B and 0 <= host <= size - 4 * B
    for t, dt, n in ((ids, torch.int32, B), (sampled, torch.int32, B), (counter, torch.int64, 1),
                     (position, torch.int64, 1), (turn, torch.int32, 2)):
        assert t.dtype == dt and t.is_contiguous() and t.numel() == n and t.is_cuda
    check(hipk().step_stage(a.args[0], a.args[1], b.args[1], a.args[2], a.table, ids.data_ptr(), sampled.data_ptr(), src // 4,
                            host // 4, B, counter.data_ptr(), position.data_ptr(), turn.data_ptr(), stream_ptr(ids)),
          "step_stage")


def step_begin(ids: torch.Tensor, src: torch.Tensor, sampled: torch.Tensor, host: torch.Tensor,
               counter: torch.Tensor, position: torch.Tensor) -> None:
    """The tokens a decode step starts from, into ``ids``: ``sampled[src]``, or ``host`` where src is
    negative (all int32 [B], src int64); then position = counter, counter += 1 (int64 [1]).  A src of
    B or more is an error on the CPU and the token -1 on the GPU."""
    if not on_gpu(ids):
        ids.copy_(torch.where(src >= 0, sampled.index_select(0, src.clamp(min=0)), host))
        position.copy_(counter)
        counter.add_(1)
        return
    B = ids.numel()
    for t, dt, n in ((ids, torch.int32, B), (src, torch.int64, B), (sampled, torch.int32, B),
                     (host, torch.int32, B), (counter, torch.int64, 1), (position, torch.int64, 1)):
        assert t.dtype == dt and t.is_contiguous() and t.numel() == n and t.is_cuda
    check(hipk().step_begin(ids.data_ptr(), src.data_ptr(), sampled.data_ptr(), host.data_ptr(), B,
                            counter.data_ptr(), position.data_ptr(), stream_ptr(ids)), "step_begin")
