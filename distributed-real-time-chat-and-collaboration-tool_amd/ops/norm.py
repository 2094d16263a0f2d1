"""Norms.  RMSNorm (+ fused residual add): csrc/kernels/norm_act_rope.hip; on a 32-bit residual
stream (+ fused residual add or embedding lookup) Dynamic Tanh: csrc/kernels/norm_dyt.hip, and RMS
norms in groups: csrc/kernels/norm_group.hip."""
from __future__ import annotations

import os

import torch

from ._ext import check, hipk, on_gpu, ptr, stream_ptr
from .gemm import Parts


def rmsnorm_ref(x: torch.Tensor, w: torch.Tensor, eps: float, gemma: bool = False,
                residual: torch.Tensor | None = None) -> torch.Tensor:
    """fp32 PyTorch reference.  With ``residual`` the sum x + residual is
    rounded to the activation dtype, written back into ``residual`` and
    normalised (the HF pre-norm residual stream semantics)."""
    if residual is not None:
        s = (x.float() + residual.float()).to(residual.dtype)
        residual.copy_(s)
        x = s
    xf = x.float()
    r = torch.rsqrt(xf.pow(2).mean(-1, keepdim=True) + eps)
    ww = w.float() + (1.0 if gemma else 0.0)
    return (xf * r * ww).to(x.dtype)


def rmsnorm(x: torch.Tensor, w: torch.Tensor, eps: float, gemma: bool = False,
            residual: torch.Tensor | None = None,
            out: torch.Tensor | None = None) -> torch.Tensor:
    """out = norm(x [+ residual]) * w (Gemma: * (1 + w)); x: [rows, H]."""
    if not on_gpu(x):
        r = rmsnorm_ref(x, w, eps, gemma, residual)
        if out is not None:
            out.copy_(r)
            return out
        return r
    assert x.dim() == 2 and x.dtype == torch.bfloat16 and x.stride(1) == 1
    rows, H = x.shape
    assert w.shape == (H,) and w.dtype == torch.bfloat16 and w.is_contiguous()
    assert H % 8 == 0 and H <= 8192 * 2
    if out is None:
        out = torch.empty((rows, H), dtype=x.dtype, device=x.device)
    assert out.stride(1) == 1 and out.shape == (rows, H)
    res_stride = 0
    if residual is not None:
        assert residual.shape == (rows, H) and residual.stride(1) == 1
        res_stride = residual.stride(0)
    check(hipk().rmsnorm(out.data_ptr(), ptr(residual), x.data_ptr(), w.data_ptr(),
                         rows, H, float(eps), x.stride(0), out.stride(0), res_stride,
                         bool(gemma), stream_ptr(x)), "rmsnorm")
    return out


def rmsnorm_parts(x: Parts, w: torch.Tensor, eps: float, gemma: bool, residual: torch.Tensor) -> torch.Tensor:
    """``rmsnorm`` of the sum of x's parts and the residual, without rounding the sum in between."""
    S, rows, H = x.slab.shape
    assert w.shape == (H,) and w.dtype == torch.bfloat16 and w.is_contiguous() and H % 8 == 0 and H <= 8192 * 2
    assert residual.shape == (rows, H) and residual.stride(1) == 1 and residual.dtype == torch.bfloat16
    out = torch.empty((rows, H), dtype=torch.bfloat16, device=residual.device)
    check(hipk().rmsnorm_parts(out.data_ptr(), residual.data_ptr(), x.slab.data_ptr(), S, w.data_ptr(), rows, H,
                               float(eps), out.stride(0), residual.stride(0), bool(gemma), stream_ptr(residual)),
          "rmsnorm_parts")
    return out


def embed(ids: torch.Tensor, table: torch.Tensor) -> torch.Tensor:
    """table[ids] of token ids [rows] (int32 or int64)."""
    if not (on_gpu(table) and ids.device == table.device and ids.dim() == 1 and ids.is_contiguous()
            and ids.dtype in (torch.int32, torch.int64) and table.dtype == torch.bfloat16
            and table.is_contiguous() and table.shape[1] % 8 == 0
            and not (table.requires_grad and torch.is_grad_enabled())):
        return torch.nn.functional.embedding(ids, table)
    out = table.new_empty(ids.shape[0], table.shape[1])
    check(hipk().embed(out.data_ptr(), ids.data_ptr(), int(ids.dtype == torch.int64), table.data_ptr(),
                       ids.shape[0], *table.shape, stream_ptr(table)), "embed")
    return out


def dyt_ref(h, w, b, alpha, y=None, ids=None, embed=None, dtype=torch.bfloat16):
    if ids is not None:
        h.copy_(embed[ids.long()])
    elif y is not None:
        h += y.float()
    return (torch.tanh(alpha * h) * w + b).to(dtype)


def dyt(h: torch.Tensor, w: torch.Tensor, b: torch.Tensor, alpha: float,
        y: torch.Tensor | None = None, ids: torch.Tensor | None = None,
        embed: torch.Tensor | None = None, dtype=torch.bfloat16) -> torch.Tensor:
    """tanh(alpha h) w + b of the 32-bit residual stream h [rows, W], after h += y (the
    preceding sublayer's output) or h = embed[ids]; h is updated in place.  w, b: float32."""
    if not on_gpu(h):
        return dyt_ref(h, w, b, alpha, y, ids, embed, dtype)
    rows, W = h.shape
    if isinstance(y, Parts):
        if dtype == torch.bfloat16 and W % 8 == 0:
            S = y.slab.shape[0]
            assert y.shape == (rows, W) and ids is None and h.is_contiguous() and w.is_contiguous() and b.is_contiguous()
            assert h.dtype == w.dtype == b.dtype == torch.float32 and w.numel() == b.numel() == W
            out = torch.empty((rows, W), dtype=dtype, device=h.device)
            check(hipk().dyt_parts(out.data_ptr(), h.data_ptr(), y.slab.data_ptr(), S, w.data_ptr(), b.data_ptr(),
                                   float(alpha), rows, W, stream_ptr(h)), "dyt_parts")
            return out
        y = y.tensor()
    assert h.dtype == w.dtype == b.dtype == torch.float32 and h.is_contiguous()
    assert w.numel() == b.numel() == W and w.is_contiguous() and b.is_contiguous()
    assert y is None or (y.shape == (rows, W) and y.stride(1) == 1 and y.dtype == dtype)
    assert ids is None or (ids.dtype == torch.int32 and ids.numel() == rows and ids.is_contiguous()
                           and embed.is_contiguous() and embed.dtype == dtype
                           and embed.shape[1] == W)
    out = torch.empty((rows, W), dtype=dtype, device=h.device)
    check(hipk().dyt(int(dtype == torch.float32), out.data_ptr(), h.data_ptr(), ptr(y),
                     y.stride(0) if y is not None else 0, ptr(ids), ptr(embed), w.data_ptr(),
                     b.data_ptr(), float(alpha), rows, W, stream_ptr(h)), "dyt")
    return out


def group_rms(h: torch.Tensor, w: torch.Tensor, groups: int, eps: float,
              y: torch.Tensor | None = None, scale: torch.Tensor | None = None,
              ids: torch.Tensor | None = None, embed: torch.Tensor | None = None,
              embed_scale: float = 1.0, width: int | None = None,
              dtype=torch.bfloat16) -> torch.Tensor:
    """RMS norm of the ``groups`` equal parts of each row of the 32-bit residual stream h [rows,
    W], times w, after h += scale * y (the preceding sublayer's output, a factor per column; more
    columns of y are ignored) or h = embed_scale * embed[ids]; h is updated in place.  w, scale:
    float32.  ``width`` > W: the output has that many columns, zeros behind the first W."""
    rows, W = h.shape
    N = width or W
    if not on_gpu(h):
        if ids is not None:
            h.copy_(embed[ids.long()].float() * embed_scale)
        elif y is not None:
            h += y[:, :W].float() * scale
        g = h.view(rows, groups, -1)
        n = (g / torch.sqrt(g.pow(2).mean(-1, keepdim=True) + eps)).view(rows, W) * w
        return torch.nn.functional.pad(n, (0, N - W)).to(dtype)
    assert h.dtype == w.dtype == torch.float32 and h.is_contiguous() and w.is_contiguous()
    assert w.numel() == W and W % groups == 0 and N >= W
    assert y is None or (y.shape[0] == rows and y.shape[1] >= W and y.stride(1) == 1
                         and y.dtype == dtype and scale.dtype == torch.float32
                         and scale.numel() == W and scale.is_contiguous())
    assert ids is None or (ids.dtype == torch.int32 and ids.numel() == rows and ids.is_contiguous()
                           and embed.is_contiguous() and embed.dtype == dtype
                           and embed.shape[1] == W)
    out = torch.empty((rows, N), dtype=dtype, device=h.device)
    check(hipk().group_rms(int(dtype == torch.float32), dict(
        out=out.data_ptr(), ldo=N, h=h.data_ptr(), y=ptr(y), ldy=y.stride(0) if y is not None else 0,
        s=ptr(scale), ids=ptr(ids), embed=ptr(embed), embed_scale=float(embed_scale),
        w=w.data_ptr(), W=W, groups=groups, eps=float(eps), rows=rows), stream_ptr(h)), "group_rms")
    return out


ROUTER_FUSE_MAX_M = 256  # rows: each reads the router's E rows again
_fuse_router = os.environ.get("DRTC_FUSED_ROUTER", "1") != "0"


def router_fusable(x: torch.Tensor | Parts, residual: torch.Tensor, router: torch.Tensor) -> bool:
    """Whether the norm ahead of a mixture also computes its router's logits: decode batches and 9 to 32
    experts (up to 8, every batch takes the same kernel: ``router_logits``) of up to 4096 columns."""
    rows, H = residual.shape
    return (_fuse_router and on_gpu(residual) and residual.dtype == router.dtype == x.dtype == torch.bfloat16
            and 1 <= rows <= ROUTER_FUSE_MAX_M and 9 <= router.shape[0] <= 32 and router.shape[1] == H
            and router.is_contiguous() and H % 8 == 0 and H <= 4096 and x.shape == residual.shape
            and residual.stride(1) == 1 and residual.stride(0) % 8 == 0
            and (isinstance(x, Parts) or x.stride(1) == 1 and x.stride(0) % 8 == 0))


class PendingNorm:
    """A pre-norm sublayer input whose RMSNorm has not run yet: norm(x [+
    residual]) * w.  The consumer either fuses the norm into its projection
    (``ops.norm_linear``: small decode batches, csrc/kernels/gemv.hip) or
    calls ``materialize()`` for the plain normalised tensor.  Either way
    ``stream()`` afterwards is the post-add residual stream h = x + residual
    (x itself when there is no residual), which the next PendingNorm adds to.
    """

    __slots__ = ("x", "residual", "w", "eps", "gemma", "_h", "_out", "pc")

    def __init__(self, x: torch.Tensor | Parts, residual: torch.Tensor | None, w: torch.Tensor,
                 eps: float, gemma: bool, pc=None):
        """``x``: a tensor, or the K slices' sums of the product ahead, which the norm adds up (needs a
        residual).  ``pc``: a ParallelContext when ``x`` is still a tensor-parallel PARTIAL
        sum: materialize() then runs the all-reduce fused with the residual add
        and the norm (ParallelContext.reduce_norm)."""
        self.x, self.residual, self.w, self.eps, self.gemma = x, residual, w, eps, gemma
        self.pc = pc
        self._h: torch.Tensor | None = None
        self._out: torch.Tensor | None = None

    @classmethod
    def done(cls, out: torch.Tensor, h: torch.Tensor, w: torch.Tensor, eps: float) -> PendingNorm:
        """The norm ``out`` of the stream ``h``, computed by the op ahead."""
        p = cls(h, None, w, eps, False)
        p._out, p._h = out, h
        return p

    def applied(self, h: torch.Tensor) -> None:
        """Record that a fused consumer computed h = x (+ residual)."""
        self._h, self.x, self.residual = h, h, None

    def materialize(self) -> torch.Tensor:
        if self._out is None:
            res = self.residual
            if self.pc is not None:
                self._out = self.pc.reduce_norm(self.x, res, self.w, self.eps, self.gemma)
                self.pc = None
            elif isinstance(self.x, Parts):
                self._out = rmsnorm_parts(self.x, self.w, self.eps, self.gemma, res)
            else:
                self._out = rmsnorm(self.x, self.w, self.eps, self.gemma, residual=res)
            self._h = res if res is not None else self.x  # rmsnorm updated res in place
            self.x, self.residual = self._h, None
        return self._out

    def materialize_router(self, router: torch.Tensor) -> tuple[torch.Tensor, torch.Tensor | None]:
        """``materialize()`` and the router logits [rows, E] in fp32 of the normalised rows, computed by the norm;
        None where it does not (``router_fusable``)."""
        x, res = self.x, self.residual
        if self._out is not None or self.pc is not None or res is None or self.gemma or not router_fusable(x, res, router):
            return self.materialize(), None
        parts = isinstance(x, Parts)
        rows, H = res.shape
        E = router.shape[0]
        out = torch.empty((rows, H), dtype=res.dtype, device=res.device)
        logits = torch.empty((rows, E), dtype=torch.float32, device=res.device)
        src, stride = (x.slab, 0) if parts else (x, x.stride(0))
        check(hipk().rmsnorm_router(out.data_ptr(), res.data_ptr(), src.data_ptr(), x.slab.shape[0] if parts else 0,
                                    self.w.data_ptr(), router.data_ptr(), logits.data_ptr(), E, rows, H, float(self.eps),
                                    stride, out.stride(0), res.stride(0), stream_ptr(res)), "rmsnorm_router")
        self._out, self._h = out, res  # updated in place
        self.x, self.residual = res, None
        return out, logits

    def stream(self) -> torch.Tensor:
        if self._h is None:
            self.materialize()
        return self._h

    def select_rows(self, idx: torch.Tensor) -> None:
        """Keep only the rows ``idx`` (int64) of every tensor this input holds:
        the last layer of a prefill pass continues with each sequence's last
        token only once its attention has read (and cached) every position."""
        if self._out is not None:
            self._out = self._out.index_select(0, idx)
        if self._h is not None:  # x is _h (materialize / applied alias them)
            self._h = self.x = self._h.index_select(0, idx)
            return
        self.x = self.x.index_select(0, idx)
        if self.residual is not None:
            self.residual = self.residual.index_select(0, idx)
