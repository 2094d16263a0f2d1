"""Projection GEMMs: one table-driven router over the hand kernels and tuned hipBLASLt.

``linear(x, w)`` computes ``x @ w.T`` (bf16, fp32 accumulate).  Every call resolves its
shape (M, N, K, row stride of x) ONCE to a route, cached per shape (``route``):

  kind      kernel                                          taken for
  "w4"      gemm_w4.hip: 4-wave hand-scheduled MFMA GEMM,   prefill-sized passes (M >= W4_MIN_M,
            persistent, 256 x 256 tiles (``mfma_gemm``)     K <= W4_MAX_K or ``_w4_long``)
  "skinny"  gemv.hip weight-streaming kernels (M <= 16)     decode buckets where the table (or
                                                            ``skinny_variant`` untuned) says so; one
                                                            or two rows by ``dot2_ok``
            gemm_stream.hip (variant STREAM, M <= 64)       where ``stream_ok`` says so
  "midm"    gemm_midm.hip medium-M kernel (M <= 256)        decode buckets where the table says so, short K
                                                            (``brief_ok``: 100 x fragments + slices);
                                                            K slices' sums for the op behind
                                                            (``linear_parts``): ``parts_form``
  "xd"      gemm_xd.hip: 128-row tiles, full K, tile order  decode buckets where the table says so
            partitioned by XCD (``xd_gemm``)                (full-batch qkv / o / down)
  "lt"      hipBLASLt with the per-shape measured solution  the other decode buckets, and
            (``csrc/kernels/gemm_lt.cpp``)                  prefill shapes the hand GEMM does not
                                                            take (tuned at the nearest M)
  "torch"   torch.nn.functional.linear (on the GPU:         decode buckets where the tuner measured
            hipBLASLt's heuristic pick)                     that pick fastest; CPU

The tuning table (``ops/tuned/gemm_<arch>.json``, keyed by the hipBLASLt version) holds, per
model decode shape and hipGraph batch bucket, the fastest measured choice among the library
solutions and the hand kernels (``scripts/tune_gemms.py``, ``tune_skinny.py``,
``tune_midm.py``, ``tune_prefill.py``); a bucket without an entry measured the library's
heuristic pick (torch's path) fastest.  A decode M that is not a bucket (e.g. an engine
``max_batch`` of 208) takes what the bucket above it measured (224: the bucket its hipGraph
batch would pad to), not an unmeasured guess.

The full-batch gate_up projection with its SiLU/GELU-GLU epilogue and the prefill o / down
projections with the residual add in their epilogue do not go through ``linear``: see
``norm_glu`` and ``linear_residual``.
"""
from __future__ import annotations

import functools
import json
import math
import os
import threading

import torch
import torch.nn.functional as F

from ._ext import check, hipk, on_gpu, ptr, stream_ptr

TUNED_DIR = os.path.join(os.path.dirname(os.path.abspath(__file__)), "tuned")
_lock = threading.Lock()
# (M, N, K, ldx) -> (hipBLASLt solution index or -1, skinny-kernel variant or 0,
#                   medium-M kernel K splits or 0, gemm_xd form or 0, gemm_xd gated form for
#                   a [gate; up] weight or 0): the decode buckets of the tuning table
_table: dict[tuple[int, int, int, int], tuple[int, int, int, int, int]] | None = None
# (N, K, ldx) -> sorted [(tuned M, algo, beats F.linear, beats addmm_)]: prefill entries
_prefill: dict[tuple[int, int, int], list[tuple[int, int, bool, bool]]] = {}
# (M, N, K, ldx, beta) -> algo chosen for a prefill-sized call (-1: torch's path)
_prefill_pick: dict[tuple[int, int, int, int, int], int] = {}
# (M, N, K, ldx) of entries that the weight-streaming GEMM leaves alone
_kept: set[tuple[int, int, int, int]] = set()
# (M, N, K, ldx) -> resolved route (kind, arg)
_routes: dict[tuple[int, int, int, int], tuple[str, int]] = {}
DECODE_MAX_M = 1024  # decode buckets end here; larger M are prefill (or mixed) passes
# the decode batch buckets (hipGraph captures, engine/decode_runner.py) the tuner measured
DECODE_BUCKETS = (1, 2, 4, 8, 16, 24, 32, 48, 64, 96, 128, 160, 192, 224, 256, 320, 384,
                  448, 512, 640, 768, 896, 1024)
_enabled = os.environ.get("DRTC_TUNED_GEMM", "1") != "0"
_prefill_enabled = os.environ.get("DRTC_PREFILL_TUNED", "1") != "0"
_midm_enabled = os.environ.get("DRTC_MIDM_GEMM", "1") != "0"
_xd_enabled = os.environ.get("DRTC_XD_GEMM", "1") != "0"
# tuned gemm_xd forms whose batch fits one row tile take non-temporal weight loads (each weight
# byte enters one CU once; profiles/r4aa: Llama-3-70B down at
# M = 256 159.6 -> 136.8 us, gated gate_up 265.7 -> 230.2, the 70B ask wave +5.2 %)
_xd_nt = os.environ.get("DRTC_XD_NT", "1") != "0"
# decode batches up to this many rows may take the skinny kernel: the table's choice where
# the shape was measured, skinny_variant()'s default otherwise; 0 disables it
SKINNY_MAX_M = int(os.environ.get("DRTC_SKINNY_MAX_M", "16"))
SKINNY_DEFAULT_MAX_M = 8  # untuned shapes: measured gains up to M = 8 only


def table_path(arch: str = "gfx950") -> str:
    return os.path.join(TUNED_DIR, f"gemm_{arch}.json")


def load_table(path: str | None = None) -> dict:
    """Read the tuning file: {str(hipblaslt_version): {"M,N,K,ldx": {...}}}."""
    path = path or table_path()
    if not os.path.exists(path):
        return {}
    with open(path) as f:
        return json.load(f)


def _activate() -> dict:
    """Parse the entries of the running hipBLASLt version (no GPU work; a library entry is
    registered with the native plan cache on its first use, outside graph capture)."""
    global _table
    if _table is not None:
        return _table
    with _lock:
        if _table is not None:
            return _table
        tab: dict[tuple[int, int, int, int], tuple[int, int, int, int, int]] = {}
        kept: set[tuple[int, int, int, int]] = set()
        pre: dict[tuple[int, int, int], list[tuple[int, int, bool, bool]]] = {}
        if _enabled and torch.cuda.is_available():
            ver = str(hipk().lt_version())
            for ks, e in load_table().get(ver, {}).items():
                M, N, K, ldx = (int(v) for v in ks.split(","))
                if e.get("prefill"):
                    if _prefill_enabled:
                        pre.setdefault((N, K, ldx), []).append(
                            (M, int(e["algo"]), bool(e.get("beta0")), bool(e.get("beta1"))))
                    if not e.get("xd"):
                        continue
                    # a prefill-table shape that is also a decode batch above the buckets
                    # (Gemma-2B's 2048 rows) with a measured gemm_xd winner: the gemm_xd form
                    # only (its library algo stays with the prefill table)
                    tab[(M, N, K, ldx)] = (-1, 0, 0, int(e["xd"]), 0)
                    continue
                nt_tuned = bool(e.get("nt_tuned"))
                tab[(M, N, K, ldx)] = (int(e.get("algo", -1)), int(e.get("skinny", 0)),
                                       int(e.get("midm", 0)) if _midm_enabled else 0,
                                       _xd_policy(M, int(e.get("xd", 0)), nt_tuned),
                                       _xd_policy(M, int(e.get("xd_glu", 0)), nt_tuned))
                if e.get("stream") == 0:
                    kept.add((M, N, K, ldx))
        for v in pre.values():
            v.sort()
        _prefill.clear()
        _prefill.update(pre)
        _kept.clear()
        _kept.update(kept)
        _prefill_pick.clear()
        _routes.clear()
        _table = tab
    return _table


def xd_nt_ok(M: int, form: int) -> bool:
    """Whether ``form`` (plain) has a non-temporal build and M fits one of its row tiles."""
    mt, nf, _ = xd_form(form)
    return form < 1000 and (mt, nf) in XD_NT_TILES and M <= XD_ROWS[mt]


def _xd_policy(M: int, form: int, nt_tuned: bool = False) -> int:
    """A tuned gemm_xd form as the router runs it (0: none / gemm_xd disabled).  An entry the
    tuner measured with the non-temporal forms among its candidates (``nt_tuned``: the
    profiles/r4ab re-tune, M = 128-256) runs exactly the form it picked - a plain winner
    stays plain; a plain form picked before the nt forms existed takes its nt twin where the
    batch fits one row tile.  DRTC_XD_NT=0 runs every form plain (an nt pick included)."""
    if not (_xd_enabled and form):
        return 0
    if not _xd_nt:
        return form % 1000
    if not nt_tuned and xd_nt_ok(M, form):
        return form + 1000
    return form


def reset() -> None:
    """Forget the activated table and every resolved route (tests / after re-tuning)."""
    global _table
    with _lock:
        _table = None
        _routes.clear()
        _parts_forms.clear()


def set_enabled(on: bool) -> None:
    global _enabled
    _enabled = bool(on)
    reset()


# ------------------------------------------------------------------ routing
def _decode_entry(M: int, N: int, K: int,
                  ldx: int) -> tuple[int, tuple[int, int, int, int, int]] | None:
    """(tuned bucket, entry) for a decode-sized shape, None for torch's (hipBLASLt heuristic)
    path.  The tuner measured every (model shape, DECODE_BUCKETS M) and kept an entry only
    where something beat the heuristic pick, so a bucket without an entry means "the
    heuristic".  A non-bucket M takes what its bucket above - the bucket the hipGraph of that
    batch would pad to - measured."""
    tab = _activate()
    ent = tab.get((M, N, K, ldx))
    if ent is not None:
        return M, ent
    if M in DECODE_BUCKETS:
        return None
    Mt = next((b for b in DECODE_BUCKETS if b >= M), None)
    if Mt is None:
        return None
    ent = tab.get((Mt, N, K, ldx))
    return (Mt, ent) if ent is not None else None


def _prefill_algo(M: int, N: int, K: int, ldx: int, beta: int) -> int:
    """Solution for a prefill-sized library GEMM: the entry tuned at the M nearest to this one
    (log scale, within 2x) for the same (N, K, ldx), if it beat torch's pick for this beta;
    -1 = use torch's path.  The native plan is per exact M (registered on first use, outside
    graph capture: prefill passes run eagerly)."""
    key = (M, N, K, ldx, beta)
    algo = _prefill_pick.get(key)
    if algo is not None:
        return algo
    algo = -1
    cands = _prefill.get((N, K, ldx))
    if cands and M > DECODE_MAX_M:
        Mt, a, b0, b1 = min(cands, key=lambda c: abs(math.log(c[0] / M)))
        if (b1 if beta else b0) and abs(math.log(Mt / M)) <= math.log(2.0):
            with _lock:
                if hipk().lt_set_algo(M, N, K, ldx, N, a) == 0:
                    algo = a
    _prefill_pick[key] = algo
    return algo


def _resolve(M: int, N: int, K: int, ldx: int) -> tuple[str, int]:
    tab = _activate()
    ent = tab.get((M, N, K, ldx))
    if M > DECODE_MAX_M and ent is not None and _xd_big_m and ent[3] and xd_supported(M, N, K, ent[3]):
        # a decode batch above the 1024 buckets with a measured gemm_xd winner (Gemma-2B's
        # 2048: qkv / o / down, profiles/r6ak)
        return ("xd", ent[3])
    if M > DECODE_MAX_M and ent is not None and ent[0] >= 0:
        # a decode batch above the 1024 buckets that was tuned as such (Gemma-2B's 2048)
        with _lock:
            if hipk().lt_set_algo(M, N, K, ldx, N, ent[0]) == 0:
                return ("lt", ent[0])
    if M > DECODE_MAX_M:
        if w4_shape_ok(M, N, K):
            # 256 x 256 tiles for a quarter of the CUs at most, or a half: smaller ones (4096 rows, 2048 x 2048 39.1 / 31.3 us,
            # 2048 x 7168 134 / 99; 2000 sizes 1.1 .. 2.9 times, 1.5 .. 2 of them where an XCD has more tiles than another), but for
            # 120 and 128 tiles of up to four columns, the same number to each XCD (8159 rows, 1024 x 8192 134 / 163)
            tiles = -(-M // 256) * (N // 256)
            form = 141 if tiles <= 64 else 241 if tiles <= 128 and (N > 1024 or tiles < 116 or tiles % 8) else 0
            if form and _xd_enabled and xd_supported(M, N, K, form):
                return ("xd", form)
            return ("w4", 0)
        a = _prefill_algo(M, N, K, ldx, 0)
        if a >= 0:
            return ("lt", a)
        full = full_form(M, N, K)
        if full and ldx % 8 == 0:
            return ("xd", full)
        return ("w4", 0) if _w4_long(M, N, K) else ("torch", 0)
    if dot2_ok(M, N, K, ldx):
        return ("skinny", 1)
    tall = tall_form(M, N, K)
    if tall and ldx % 8 == 0:
        return ("xd", tall)
    found = _decode_entry(M, N, K, ldx)
    wide = wide_form(M, N, K)
    if wide and not (found is not None and found[1][3]):  # (entries of gemm_xd: measured against its other forms)
        return ("xd", wide)
    small = small_form(M, N, K)
    if small and ldx % 8 == 0:
        return ("xd", small)
    if brief_ok(M, N, K) and ldx % 8 == 0 and brief_pays(M, N, K, found is not None and found[1][0] >= 0):
        return ("midm", 201)
    # the rule goes ahead of the table, but for entries that were measured faster ("stream": 0)
    if ldx % 8 == 0 and stream_ok(M, N, K) and (found is None or (found[0], N, K, ldx) not in _kept):
        return ("skinny", STREAM)
    if found is None:
        form = deep_form(M, N, K) or full_form(M, N, K)
        if form and ldx % 8 == 0:
            return ("xd", form)
        v = skinny_variant(M, N, K, ldx)
        return ("skinny", v) if v else ("torch", 0)
    _, (algo, sk, midm, xd, _) = found
    if K <= 1024 and not (sk or midm or xd) and ldx % 8 == 0 and full_form(M, N, K):
        return ("xd", full_form(M, N, K))
    if algo < 0 and not (sk or midm or xd):
        return ("torch", 0)  # measured: the library's heuristic pick beat every candidate
    if sk and M <= SKINNY_MAX_M and skinny_supports(sk, M, N, K, ldx):
        return ("skinny", sk)
    if xd and xd_supported(M, N, K, xd):
        return ("xd", xd)
    if midm and midm_supported(M, N, K):
        return ("midm", midm)
    if algo >= 0:
        with _lock:  # the native plan is per exact M: validate the solution at this M
            if hipk().lt_set_algo(M, N, K, ldx, N, algo) == 0:
                return ("lt", algo)
    v = skinny_variant(M, N, K, ldx)
    return ("skinny", v) if v else ("torch", 0)


def small_form(M: int, N: int, K: int) -> int:
    """gemm_xd form of 64-row tiles for a plain product of 17 .. 256 rows that they cut into at most a workgroup a CU, of
    32 columns or else 64: what a workgroup reads, at 45 - 65 GB/s, is the time of such a product, and its other forms and
    the library's leave half the chip idle or read all rows everywhere.  us, the best of those / this: 3584 x 2048, 64 rows
    9.5 / 7.7, 128 10.9 / 7.8, 224 10.7 / 8.9; 2048 x 2048, 224 10.5 / 7.8; 3840 x 2048, 100 14.0 / 8.2; 6912 x 4096, 32 15.5 / 13.6,
    100 20.3 / 18.9; 12800 x 4096, 32 23.7 / 19.7, 64 25.3 / 23.4; 4096 x 4096, 160 19.7 / 17.5.
    Not where K slices fill the chip better: long K on half the CUs (4096 x 4096, 64 rows 14.3 / 16.8), nor for long K and
    whole row tiles, several of them (6144 x 4096, 100 rows 20.1 / 18.6, 128 20.8 / 21.1), nor 64 columns
    where up to 32 rows stream (8448 x 2048, 32 rows 12.2 / 13.6).  Weights of 32 MiB on, one row tile: non-temporal (6912 x 4096, 64 rows 18.6 /
    17.1; 8192 x 2048 11.8 / 10.1; 3840 x 2048 9.4 / 9.7)."""
    if not (_xd_enabled and _enabled and 17 <= M <= 256 and 2048 <= K <= 4096 and N >= 2048):
        return 0
    tiles = -(-M // 64)
    nf = next((n for n in (1, 2) if N % (32 * n) == 0 and tiles * (N // (32 * n)) <= 256), 0)
    items = tiles * (N // (32 * nf)) if nf else 0
    if not nf or (K > 2048 and (items < 160 or M > 64 and (M - 1) % 64 >= 48)) or (
            nf == 2 and M <= 32 and stream_ok(M, N, K)):
        return 0
    form = 10 * nf + 1 + (1000 if _xd_nt and tiles == 1 and N * K >= 1 << 24 else 0)
    return form if xd_supported(M, N, K, form) else 0


def dot2_ok(M: int, N: int, K: int, ldx: int) -> bool:
    """Whether one or two rows go to the dot2 kernel ahead of the table, whose entries were measured before its
    weights went past the caches.  us, the MFMA form or the library / this: one row 32000 x 4096 43.7 / 40.5, 64128 x
    4096 83.2 / 77.9, 128256 x 2048 82.8 / 76.9, 256000 x 2048 162 / 152, 57344 x 8192 157 / 143, 128256 x 8192 346 / 314;
    two rows 16384 x 4096 24.1 / 22.2, 32000 x 4096 43.3 / 39.3, 57344 x 8192 154 / 134.  Smaller products gain less (two rows of
    8192 x 2048 8.3 / 8.3, 4096 x 3584 8.2 / 7.8, 3584 x 2048 5.5 / 5.7) and stay with the table."""
    return _enabled and M <= min(2, SKINNY_MAX_M) and N * K >= 1 << 25 and skinny_supports(1, M, N, K, ldx)


def brief_ok(M: int, N: int, K: int) -> bool:
    """Whether gemm_midm takes a product of a few K tiles in one slice and 64 columns to a workgroup: all of it is
    launch, one round trip and the store."""
    return (_midm_enabled and _enabled and K % 64 == 0 and K <= 256 and 17 <= M <= 256 and M * K <= 32768
            and N % 64 == 0 and 1024 <= N <= 8192)


def brief_pays(M: int, N: int, K: int, listed: bool) -> bool:
    """... and is the faster kernel for it, against the library's pick or (``listed``) the table's.  us, the pick /
    this: 1024 x 64, 17 rows 3.5 / 2.9, 64 3.6 / 3.3; 2560 x 128, 17 rows 4.0 / 3.2, 64 4.2 / 3.8, 80 4.0 / 4.2, 112 4.4 / 4.7;
    5120 x 256, 64 rows 5.4 / 4.7, 112 5.7 / 5.9, 128 6.2 / 6.1; 3072 x 192, 72 rows 0.92 of it, 128 0.94.  It reads all rows in
    every workgroup, so many of them lose: 1024 x 128, 160 rows 3.7 / 4.9, 256 3.7 / 6.5.  The table's, 2048 x 128: 48 rows 6.2 /
    3.5, 128 6.3 / 4.6, 200 7.0 / 5.8, 256 6.8 / 6.4; 4096 x 256, 48 rows 6.5 / 4.5, 128 5.9 / 6.0."""
    return M <= 64 or M <= 128 and N * K >= 3072 * 192 or listed


def tall_form(M: int, N: int, K: int, glu: bool = False, act: str = "silu") -> int:
    """gemm_xd form of one row tile of 160, 192 or 224 rows for a product of 129 .. 224 rows (N output columns, gated: of a
    half) that tiles of 128 rows of W cut into one well filled round of the CUs; 160 rows also where tiles of 64 do, nearly
    full.  Other forms pad the rows to 256, or read W twice.  us, the best of them / this: 28672 x 4096 gated, 132 rows
    58.4 / 48.0, 160 56.9 / 50.9, 192 56.2 / 54.2, 224 57.8 / 57.7; 32000 x 4096, 144 rows 60.6 / 53.1, 208 61.0 / 58.4; 32000 x
    2048, 160 33.4 / 30.3; 25600 x 4096, 224 57.2 / 54.2; 20480 x 2048 (160 tiles), 160 28.2 / 26.4, 224 30.0 / 29.2; in tiles of
    64: 14336 x 2048 gated, 132 rows 22.3 / 18.3, 160 20.4 / 19.4, 12800 x 2048 20.1 / 19.0, 16384 x 4096 gated 39.1 / 36.7.
    More than a round: 57344 x 4096 gated, 176 rows 100.6 / 109; fewer tiles: 16384 x 4096 gated, 160 rows 39.1 / 48.4, and of 64
    8448 x 2048, 160 rows 17.6 / 17.9; 192 rows in tiles of 64 12800 x 2048 21.5 / 21.4.  Tiles of 64 where the others' rows of W are
    multiples of 4 KB apart, or long: over 3300 sizes K 2048, 4096, 6144, 8192 1.06, 1.07, 1.02, 1.18, 11008 and 14336 1.06 and 1.11, but
    2304 .. 3584 0.96, 5120 0.91, 7168 0.98 (13312 x 5120 gated, 148 rows 40.5 / 46.3)."""
    if not (129 <= M <= 224 and K >= 2048 and _xd_enabled and _enabled and _xd_nt):
        return 0
    mt, rows = 3 if M <= 160 else 4 if M <= 192 else 5, 2 * N if glu else N
    nf = 4 if rows % 128 == 0 and 160 <= rows // 128 <= 256 else 0
    if not nf and mt == 3 and rows % 64 == 0 and 192 <= rows // 64 <= 256 and (K % 2048 == 0 or K > 8192):
        nf = 2
    if not nf or act == "clamped" and nf not in XD_CLAMP_NF:
        return 0
    form = 1001 + 100 * mt + 10 * nf
    return form if xd_supported(M, N, K, form, glu) else 0


DEEP_FORMS = (122, 123, 124, 142, 143, 144, 162, 163, 164, 242, 243, 244)


@functools.lru_cache(maxsize=4096)
def _deep_form(M: int, N: int, K: int) -> int:
    best, cost = 0, 0.0
    for form in DEEP_FORMS:
        mt, nf, sk = xd_form(form)
        tm, tn = XD_ROWS[mt], 32 * nf
        items = -(-M // tm) * (N // tn) * sk
        if not 100 <= items <= 256 or not xd_supported(M, N, K, form):
            continue
        us = 7 + (tm + tn) * K / sk / 1e6 * (20 + 0.0387 * items) + tm * tn / 1e5 * (31 + 1.1 * (sk - 1))
        if not best or us < cost:
            best, cost = form, us
    return best


def deep_form(M: int, N: int, K: int) -> int:
    """gemm_xd form, K in slices, of a product of 257 .. 1024 rows without a tuned one that has long K and too few tiles for
    the CUs, which the library takes whole: the form of least cost by a fit (us; 6 to 9 % off) of the bytes a workgroup reads, those that
    all of them do and the slices' sums.  us, library / this: 2048 x 7168, 257 rows 28.5 / 23.0, 512 32.0 / 28.3, 640 40.2 / 35.4,
    1024 45.9 / 42.5; 2048 x 14336, 448 rows 58.8 / 40.8; 1024 x 7168, 1024 32.4 / 27.5; 2304 x 9216 1.24 times, 5120 x 13824 1.26, 4096 x
    11008 1.17 over thirteen row counts.  Shorter K: 2048 x 4096, 768 rows 24.1 / 26.9; three of the library's row tiles of
    256 on wider W: 4096 x 7168, 768 rows 54.9 / 57.7, 4096 x 8192 57.9 / 61.0."""
    if not (257 <= M <= DECODE_MAX_M and K >= 5632 and _xd_enabled and _enabled) or 640 < M <= 768 and N >= 4096 and K <= 8192:
        return 0
    return _deep_form(M, N, K)


def full_form(M: int, N: int, K: int) -> int:
    """gemm_xd form of a plain product of 129 .. 3072 rows without a tuned one that some tile, the smallest that makes at
    most a workgroup a CU, cuts into one well filled round: 200 workgroups, 128 where K is short.  420 sizes of 24 widths, K 512
    .. 5120, the library's time / this: 200 .. 256 workgroups 1.31 (K 512, 768), 1.20 (to 1536), 1.21 (2048), 1.13 (to 3072), 1.11, nine
    of 203 below 0.97; K to 1536, 128 .. 199 1.27; longer K and fewer 1.06, a third below 0.97.  us: 6656 x 2048, 256 rows 24.7 /
    16.9, 448 24.4 / 19.9, 1024 31.1 / 29.6; 12800 x 4096, 256 49.4 / 42.8; 3072 x 2048, 1088 23.6 / 19.1; past 3072 rows 3072 x 2048,
    3360 37.7 / 39.9, 1024 x 3072, 4064 28.3 / 33.0.  The table's library solutions of short K as well: 4096 x 512, 256 rows 8.2 /
    5.5, 1024 9.7 / 8.6.
    Longer K, over 28,000 sizes of 30 widths: 5120 .. 7168 1.09, longer 1.08; left to the library where a class of them loses:
    K above 7168 with less than three quarters of the tiles' rows used, but in 64 columns (0.87 in tiles of 256 x 128, 0.96 of 128 x 128; 12800
    x 12800, 261 rows 130.8 / 183.8, of 300 rows at K 7168 1.01, from 385 rows on 1.13), tiles of 256 x 192 with less than four
    fifths (0.93 .. 1.02), 64 columns past 2048 rows (K to 5120 0.98, longer 0.95 .. 0.84)."""
    if not (129 <= M <= 3072 and _xd_enabled and _enabled):
        return 0
    for form in (121, 141, 161, 241, 261):
        mt, nf, _ = xd_form(form)
        rows = -(-M // XD_ROWS[mt])
        items = rows * (N // (32 * nf))
        if items <= 256 and xd_supported(M, N, K, form):
            if items < (128 if K <= 1536 else 200):
                return 0
            used = M / (rows * XD_ROWS[mt])
            if K > 7168 and nf > 2 and used < 0.75 or K > 1536 and form == 261 and used < 0.8 or K > 3072 and nf == 2 and M > 2048:
                return 0
            return form + 1000 if _xd_nt and xd_nt_ok(M, form) else form
    return 0


def wide_form(M: int, N: int, K: int) -> int:
    """gemm_xd form of a plain product of 24 .. 256 rows, one row tile, whose columns fill the CUs in whole
    rounds: vocabulary heads above all.  Each workgroup walks K from another tile (gemm_xd.hip), which neither
    the library nor the streaming GEMM does.  us, their best / this: 32000 x 2048, 24 rows 26.5 / 23.4, 64 32.6 / 24.3, 128
    33.3 / 27.2, 192 36.0 / 34.9; 32000 x 4096, 17 46.0 / 47.5, 24 47.3 / 45.9, 64 58.1 / 47.2; 64128 x 4096, 32 91.2 /
    82.7, 96 115.5 / 96.6; 128256 x 2048, 144 130 / 119; 57344 x 8192, 64 190 / 168, 192 235 / 203.  Rounds that are not
    full: 50176 columns (0.77), 32 rows 39.4 / 40.0, 192 53.4 / 53.8; 27648 (0.84) 43.9 / 35.9, 61.4 / 55.2.  Short K:
    64000 x 1024, 64 rows 27.8 / 29.3.  Above 128 rows tiles of 256 x 256, or 256 x 128 in one round (64128 columns, not a
    multiple of 256, 256 rows 126.9 / 131.2)."""
    if not (_xd_enabled and _enabled and 24 <= M <= 256 and K >= 2048):
        return 0

    def full(columns):
        tiles = N // columns
        return N % columns == 0 and tiles >= 0.84 * 256 * -(-tiles // 256)

    if M <= 128:
        form = 1141 if full(128) else 0
    else:
        form = 1281 if full(256) else 1241 if full(128) and N <= 256 * 128 else 0
    form = form if _xd_nt else form % 1000
    return form if form and xd_supported(M, N, K, form) else 0


# DRTC_XD_BIG_M=0: decode batches above DECODE_MAX_M ignore tuned gemm_xd entries (A/B knob)
_xd_big_m = os.environ.get("DRTC_XD_BIG_M", "1") != "0"


def route(M: int, N: int, K: int, ldx: int) -> tuple[str, int]:
    """The kernel ``linear`` runs for y[M, N] = x[M, K] @ W[N, K]^T with x's row stride ldx on
    the GPU: (kind, arg) as in the module docstring, resolved once per shape."""
    key = (M, N, K, ldx)
    r = _routes.get(key)
    if r is None:
        r = _resolve(M, N, K, ldx)
        _routes[key] = r
    return r


def _gpu_bf16(x: torch.Tensor, w: torch.Tensor) -> bool:
    return (on_gpu(x) and _enabled and x.dim() == w.dim() == 2 and x.dtype == torch.bfloat16
            and w.dtype == torch.bfloat16 and x.stride(1) == 1 and w.is_contiguous())


def _aligned(x: torch.Tensor, w: torch.Tensor) -> bool:
    return x.stride(0) % 8 == 0 and x.data_ptr() % 16 == 0 and w.data_ptr() % 16 == 0


def _staged(x: torch.Tensor, w: torch.Tensor) -> bool:
    """What kernels that load rows into LDS take: whole 16-byte pieces, 32-bit offsets of up to 256 rows."""
    return _aligned(x, w) and x.stride(0) < 1 << 22


def linear(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """y = x @ w.T for x [M, K] (row stride ldx), w [N, K] contiguous."""
    if not _gpu_bf16(x, w) or w.shape[1] != x.shape[1]:  # (refuses widths that differ)
        return F.linear(x, w)
    M, K = x.shape
    N = w.shape[0]
    kind, arg = route(M, N, K, x.stride(0))
    if kind == "w4" and _aligned(x, w):
        return mfma_gemm(x, w, "store", variant=_w4v(K), group_m=w4_group_m(M, N, K))
    if kind == "lt":
        y = torch.empty((M, N), dtype=x.dtype, device=x.device)
        check(hipk().lt_gemm(y.data_ptr(), x.data_ptr(), w.data_ptr(), M, N, K, x.stride(0), N,
                             0.0, stream_ptr(x)), "lt_gemm")
        return y
    if kind == "skinny" and (arg != STREAM or _aligned(x, w)):
        return skinny_linear(x, w, arg)
    if kind in ("midm", "xd") and _staged(x, w):
        if kind == "xd":
            return xd_gemm(x, w, form=arg)
        return midm_gemm(x, w, "store", splits=arg % 100, nf=arg // 100 or 4)
    return F.linear(x, w)


# ------------------------------------------------------------------ skinny decode kernels
DUAL = range(1, 10)  # skinny variants that take a second product along
# rows of W per workgroup of each MFMA variant (gemv.hip launch_skinny_gemm)
SKINNY_ROWS = {2: 16, 3: 16, 4: 32, 5: 32, 6: 16, 7: 64, 8: 128, 9: 64}


def skinny_supports(v: int, M: int, N: int, K: int, ldx: int) -> bool:
    """Whether skinny variant ``v`` covers the shape (mirrors the launcher)."""
    if not 1 <= M <= 16 or ldx % 8 or N % 4:
        return False
    if v == 1:
        return M <= 8 and K % 512 == 0
    return v in SKINNY_ROWS and K % 128 == 0 and N % SKINNY_ROWS[v] == 0


def skinny_variant(M: int, N: int, K: int, ldx: int) -> int:
    """Default skinny-kernel form for an untuned shape: 1 = VALU dot2 for M <= 2, 3 = MFMA
    (1 tile, 8 K-split waves) up to M = 8; 0 = leave it to the library."""
    if M > min(SKINNY_MAX_M, SKINNY_DEFAULT_MAX_M):
        return 0
    for v in ((1, 3) if M <= 2 else (3,)):
        if skinny_supports(v, M, N, K, ldx):
            return v
    return 0


def skinny_ok(M: int, N: int, K: int, ldx: int) -> bool:
    return skinny_variant(M, N, K, ldx) != 0


def skinny_linear(x: torch.Tensor, w: torch.Tensor, variant: int = 0) -> torch.Tensor:
    """y = x @ w.T on a skinny decode kernel (M <= 16 rows of x; STREAM: up to 64)."""
    if variant == STREAM:
        return stream_gemm(x, w)
    M, K = x.shape
    N = w.shape[0]
    variant = variant or skinny_variant(M, N, K, x.stride(0))
    y = torch.empty((M, N), dtype=x.dtype, device=x.device)
    check(hipk().skinny_gemm(y.data_ptr(), x.data_ptr(), w.data_ptr(), M, N, K, x.stride(0), N,
                             variant, 0, 0, 0, 0, 0, 0, 0, stream_ptr(x)), "skinny_gemm")
    return y


def linear_beside(x: torch.Tensor, w: torch.Tensor, x2: torch.Tensor, w2: torch.Tensor, out2: torch.Tensor | None = None,
                  relu2: bool = False) -> tuple[torch.Tensor, torch.Tensor]:
    """``linear(x, w)``, and ``linear(x2, w2)`` or (``relu2``, into ``out2``) ``squared_relu``: in one launch where both are
    products of the same K that the skinny kernels take (gemv.hip SkinnyBeside), by the first's choice of them."""
    if (_gpu_bf16(x, w) and _gpu_bf16(x2, w2) and x.shape == x2.shape and x.shape[0] <= SKINNY_MAX_M
            and w.shape[1] == w2.shape[1] == x.shape[1]):
        (M, K), N, N2 = x.shape, w.shape[0], w2.shape[0]
        v, v2 = _choice(M, N, K, x.stride(0)), _choice(M, N2, K, x2.stride(0))
        if v in DUAL and v2 in DUAL and (v == v2 or v != 1 != v2) and skinny_supports(v, M, N2, K, x2.stride(0)) and (
                out2 is None or out2.stride(1) == 1 and out2.stride(0) % 4 == 0 and out2.data_ptr() % 8 == 0):
            y = torch.empty((M, N), dtype=x.dtype, device=x.device)
            if out2 is None:
                out2 = torch.empty((M, N2), dtype=x.dtype, device=x.device)
            assert out2.shape == (M, N2) and out2.dtype == x.dtype
            check(hipk().skinny_gemm(y.data_ptr(), x.data_ptr(), w.data_ptr(), M, N, K, x.stride(0), N, v,
                                     out2.data_ptr(), x2.data_ptr(), w2.data_ptr(), N2, x2.stride(0), out2.stride(0),
                                     2 if relu2 else 0, stream_ptr(x)), "skinny_gemm")
            return y, out2
    y = linear(x, w)
    if relu2:
        return y, squared_relu(x2, w2, out2)
    y2 = linear(x2, w2)
    return y, y2 if out2 is None else out2.copy_(y2)


def _choice(M: int, N: int, K: int, ldx: int) -> int:
    """Skinny variant ``linear`` runs for this shape (0 = another kernel)."""
    kind, arg = route(M, N, K, ldx)
    return arg if kind == "skinny" else 0


# ------------------------------------------------------------------ fused forms
_fuse_residual = os.environ.get("DRTC_RESIDUAL_GEMM", "1") != "0"
# measured (scripts/residual_gemm_bench.py, MI355X, H=4096): at 16k rows the beta=1 GEMM
# costs the same as beta=0 while the following RMSNorm drops from ~90 us (read x + residual,
# write both) to ~39 us (read h, write out); at 1024 rows both norms are launch-latency
# bound (7-8 us) - no gain
RESIDUAL_FUSE_MIN_M = 4096


def residual_fusable(x: torch.Tensor, residual: torch.Tensor) -> bool:
    """Whether ``linear_residual`` pays for x [M, K] -> residual [M, N]: on the GPU at
    prefill-sized M (bf16).  Elsewhere the caller runs ``linear`` and leaves the add to the
    next fused add-RMSNorm."""
    return (_fuse_residual and on_gpu(x) and x.dim() == 2 and x.shape[0] >= RESIDUAL_FUSE_MIN_M
            and x.dtype == residual.dtype == torch.bfloat16
            and residual.dim() == 2 and residual.shape[0] == x.shape[0]
            and residual.stride(1) == 1)


def linear_residual(x: torch.Tensor, w: torch.Tensor, residual: torch.Tensor) -> torch.Tensor:
    """residual += x @ w.T with the add in the GEMM epilogue (in place into the residual
    stream), for the o / down projections of a prefill pass; returns the updated residual.
    One rounding to bf16 (of the fp32 accumulator plus the residual) instead of two."""
    assert residual.shape == (x.shape[0], w.shape[0]) and w.dtype == x.dtype
    M, K = x.shape
    N = w.shape[0]
    if w4_ok(x, w, residual):
        return mfma_gemm(x, w, "residual", residual=residual, out=residual, variant=_w4v(K),
                         group_m=w4_group_m(M, N, K))
    if (_enabled and x.stride(1) == 1 and w.is_contiguous() and residual.stride(0) == N
            and x.dtype == torch.bfloat16):
        _activate()
        if _prefill_algo(M, N, K, x.stride(0), 1) >= 0:
            check(hipk().lt_gemm(residual.data_ptr(), x.data_ptr(), w.data_ptr(), M, N, K,
                                 x.stride(0), N, 1.0, stream_ptr(x)), "lt_gemm")
            return residual
    return residual.addmm_(x, w.t())


_fuse_norm = os.environ.get("DRTC_FUSED_NORM_GEMM", "1") != "0"
# measured: the fused norm pays at M = 1 only (gemv.hip skinny_norm_gemm_kernel)
NORM_FUSE_MAX_M = 1


def _norm_fused(p, w: torch.Tensor, act: int = -1):
    """norm(p) @ w.T, gated with ``act`` >= 0, in one launch (``skinny_norm_gemm_kernel``), or None where the
    projection would not run on the skinny dot2 kernel."""
    x, res = p.x, p.residual
    if not (_fuse_norm and p._out is None and p.pc is None and isinstance(x, torch.Tensor)
            and _gpu_bf16(x, w) and p.w.is_contiguous()
            and (res is None or (res.stride(1) == 1 and res.shape == x.shape))):
        return None
    M, K = x.shape
    N = w.shape[0]
    if not (M <= (NORM_FUSE_MAX_M if act < 0 else 1) and K in (2048, 4096, 8192) and N % 4 == 0
            and x.stride(0) % 8 == 0 and (res is None or res.stride(0) % 8 == 0)
            and _choice(M, N, K, K) == 1):
        return None
    if act >= 0:
        N //= 2
    y = torch.empty((M, N), dtype=x.dtype, device=x.device)
    h = torch.empty((M, K), dtype=x.dtype, device=x.device) if res is not None else None
    check(hipk().skinny_norm_gemm(
        y.data_ptr(), ptr(h), x.data_ptr(), ptr(res), p.w.data_ptr(), w.data_ptr(), M, N,
        K, x.stride(0), res.stride(0) if res is not None else 0, K, N, float(p.eps),
        bool(p.gemma), act, stream_ptr(x)), "skinny_norm_gemm")
    p.applied(h if h is not None else x)
    return y


def norm_linear(p, w: torch.Tensor, parts: int = 0) -> torch.Tensor | Parts:
    """y = rmsnorm(p.x [+ p.residual]) @ w.T for an ``ops.PendingNorm`` p; ``parts``: or the sums of up to that
    many K slices (``linear_parts``).

    When the projection would run on the skinny dot2 kernel anyway (small decode batches,
    measured per shape) the norm is fused into it (gemv.hip ``skinny_norm_gemm_kernel``):
    one launch instead of two, and the new residual stream is written by the GEMM.
    Otherwise the norm is materialised and ``linear`` runs."""
    y = _norm_fused(p, w)
    if y is not None:
        return y
    h = p.materialize()
    return linear_parts(h, w, parts) if parts > 1 else linear(h, w)


def norm_glu_row(p, w: torch.Tensor, act: str = "silu"):
    """act(norm(p) @ gate.T) * (norm(p) @ up.T) of one row in one launch, the fused [gate; up] weight on the skinny
    dot2 kernel; None where another kernel takes the product (``norm_glu``)."""
    code = {"silu": 0, "gelu_tanh": 1}.get(act)
    return None if code is None or not _fuse_glu else _norm_fused(p, w, code)


_fuse_glu = os.environ.get("DRTC_FUSED_GLU_GEMM", "1") != "0"
GLU_FUSE_MAX_M = 1


def glu_linear(gu: torch.Tensor, w: torch.Tensor, act: str = "silu", parts: bool = False):
    """y = (act(gu[:, :I]) * gu[:, I:]) @ w.T (the down projection of a gated MLP), by ``linear`` or
    (``parts``) ``linear_parts`` behind ops.act_glu.  When the
    projection would run on the skinny dot2 kernel the activation is computed inside it while
    loading its input (gemv.hip, no act_glu launch)."""
    from .activation import act_glu

    if _fuse_glu and _gpu_bf16(gu, w) and act in ("silu", "gelu_tanh"):
        M, I2 = gu.shape
        I, N = I2 // 2, w.shape[0]
        if (M <= GLU_FUSE_MAX_M and I2 % 2 == 0 and w.shape[1] == I and I % 512 == 0
                and N % 4 == 0 and gu.stride(0) % 8 == 0 and _choice(M, N, I, I) == 1):
            y = torch.empty((M, N), dtype=gu.dtype, device=gu.device)
            check(hipk().skinny_glu_gemm(y.data_ptr(), gu.data_ptr(), w.data_ptr(), M, N, I,
                                         gu.stride(0), N, 0 if act == "silu" else 1,
                                         stream_ptr(gu)), "skinny_glu_gemm")
            return y
    return (linear_parts if parts else linear)(act_glu(gu, act), w)


# ------------------------------------------------------------------ weight-streaming decode GEMM
STREAM_MAX_M = 64
# K steps of 32 that a wave's registers hold of 16, 32 or 64 rows of x (gemm_stream.hip instances)
STREAM_KS = {1: (16, 14, 8), 2: (16, 14, 8), 4: (8,)}
STREAM_MAX_SLICES = 4  # plain products up to 32 rows
STREAM = 10  # as a variant of the skinny kernels in the router
STREAM_ACT = {"store": (0, 0), "relu2": (0, 1), "silu": (1, 0), "gelu_tanh": (1, 1), "clamped": (1, 2)}


def stream_slices(M: int, N: int, K: int, epi: str = "store") -> int:
    """K slices of ``stream_gemm`` for the shape (N output columns), 0 where it does not take it."""
    if not (1 <= M <= STREAM_MAX_M and N % 16 == 0 and N >= 16 and epi in STREAM_ACT):
        return 0
    mt = 1 if M <= 16 else 2 if M <= 32 else 4
    most = 1 if mt > 2 or STREAM_ACT[epi][0] else STREAM_MAX_SLICES
    for ks in STREAM_KS[mt]:
        s, parts = K // (256 * ks), N // 16 * mt
        if K % (256 * ks) == 0 and 1 <= s <= most and \
                (s == 1 or (s * parts * 1024 <= WS_SLAB_BYTES and parts < WS_COUNTERS - 1)):
            return s
    return 0


def stream_ok(M: int, N: int, K: int, epi: str = "store") -> bool:
    """Whether a decode batch of M rows takes ``stream_gemm``, N output columns.  us against what the
    table picks, activation pass included, both without the norm ahead (it costs the same):
      one slice, up to 16 rows: from 24 M weights on, where the stream outlasts the first loads
        (6144 x 4096 14.0 / 15.5, 14336 x 2048 gated 16.2 / 18.4, 32000 x 4096 46 / 65; 8192 x 2048 11.7 /
        10.3); two rows and one stay with the dot2 form (6144 x 4096 12.0 / 11.5)
      17 .. 32 rows: 2048 columns take what the other kernels need for 64 rows (2560 x 2048 8.1 / 11.4);
        4096 columns leave the registers for one workgroup per CU, which pays for long W (16384 rows 29 /
        33, 32000 51 / 65; 12800 27 / 26)
      33 .. 64 rows: 2048 columns and long W (64000 rows 59 / 71; 8192 15.7 / 12.6); gated where gemm_xd's
        form does not fill the chip (32768 rows 34.7, gemm_xd 32.5)
      slices: adding the parts up costs about 3 us, and more for more rows.  Plain products of two to four,
        to 8 rows (2048 x 7168 11.5 / 13.9, 8192 x 8192 28.3 / 31.8, 5120 x 12288 27.0 / 42.0; 4096 x 7168, the
        closest, 15.7 / 14.4); 9 .. 16 rows outside of the 2048 .. 5120 columns where the library's pick holds
        (4096 x 8192 17.9 / 16.6, 2560 x 8192 16.8 / 14.0; 2048 x 7168 12.4 / 12.7, 5120 x 12288 27.6 / 33.5)
        unless in four (4096 x 14336 25.2 / 27.3); above 16 rows they lose but for 32 rows of
        two slices of 14 steps (2048 x 7168 15.7 / 18.6; 28 rows 14.9 / 12.9; 2048 x 8192 17.1 / 16.1)"""
    s = stream_slices(M, N, K, epi)
    if not s or M < 3 or SKINNY_MAX_M <= 0:
        return False
    rows = N * (1 + STREAM_ACT[epi][0])
    if s > 1:
        return epi == "store" and (M <= 8 or M <= 16 and (N <= 2048 or N >= 5120 or s == 4)
                                   or M == 32 and N <= 2048 and K == 7168)
    if M <= 16:
        return rows * K >= 24_000_000
    if M <= 32:
        return rows >= (16384 if K > 2048 else 2048)
    return rows >= 14336 and not (STREAM_ACT[epi][0] and glu_form(M, rows, K, K, epi))


def stream_gemm(x: torch.Tensor, w: torch.Tensor, epi: str = "store", out: torch.Tensor | None = None,
                limit: float = 0.0) -> torch.Tensor:
    """y = epi(x @ w.T) for at most 64 rows, csrc/kernels/gemm_stream.hip: one pass over W with x in
    registers.  epi as ``xd_gemm``, without "residual"."""
    M, K = x.shape
    glu, act = STREAM_ACT[epi]
    N = w.shape[0] // 2 if glu else w.shape[0]
    s = stream_slices(M, N, K, epi)
    assert s and x.dtype == w.dtype == torch.bfloat16 and x.stride(1) == 1 and w.is_contiguous() and w.shape[1] == K
    if out is None:
        out = torch.empty((M, N), dtype=x.dtype, device=x.device)
    assert out.shape == (M, N) and out.stride(1) == 1 and out.dtype == x.dtype
    slab, cnt = gemm_workspace(x.device) if s > 1 else (None, None)
    check(hipk().stream_gemm(out.data_ptr(), x.data_ptr(), w.data_ptr(), M, N, K, x.stride(0), out.stride(0), glu, act,
                             limit, s, ptr(slab), slab.numel() * 4 if slab is not None else 0, ptr(cnt),
                             cnt.numel() if cnt is not None else 0, stream_ptr(x)), "stream_gemm")
    return out


# ------------------------------------------------------------ hand-written MFMA GEMM
EPI = {"store": 0, "residual": 1, "silu": 2, "gelu_tanh": 3, "relu2": 4, "clamped": 5}
GATED = ("silu", "gelu_tanh", "clamped")  # activations with a fused [gate; up] epilogue
_ws_lock = threading.Lock()
_ws: dict[int, tuple[torch.Tensor, torch.Tensor]] = {}
WS_SLAB_BYTES = 128 << 20   # fp32 split-K slabs (per device)
WS_COUNTERS = 1 << 16


# every split-K workspace created in this process (the shared per-device ones and the private
# ones of second streams): check_splitk_fault reads the fault word of each
_all_ws: list[tuple[torch.Tensor, torch.Tensor]] = []


# per-thread override of the device workspace: GEMMs issued inside ``private_workspace(ws)``
# (the second micro-batch stream of a decode step) use ``ws``
_ws_local = threading.local()


class private_workspace:
    """Context manager: every split-K / medium-M GEMM issued by this thread inside it takes
    ``ws`` (from ``new_gemm_workspace``) instead of the device's shared workspace - for GEMMs
    that run concurrently with the shared workspace's users on another stream."""

    def __init__(self, ws: tuple[torch.Tensor, torch.Tensor] | None):
        self.ws = ws

    def __enter__(self):
        self.prev = getattr(_ws_local, "ws", None)
        _ws_local.ws = self.ws
        return self.ws

    def __exit__(self, *exc):
        _ws_local.ws = self.prev
        return False


def gemm_workspace(dev: torch.device) -> tuple[torch.Tensor, torch.Tensor]:
    """Split-K workspace of a device: fp32 slabs + per-tile arrival counters (zeroed once;
    the last arriver of each tile re-arms its counter; the LAST counter is the fault word,
    ``check_splitk_fault``).  One per device, shared by every GEMM on the engine's stream (and
    the medium-M kernel's partial slabs); a GEMM issued concurrently on another stream passes
    its own (``ws=``, or ``private_workspace``).  Created before any graph capture (the
    engine's eager warm-up does)."""
    key = dev.index if dev.index is not None else torch.cuda.current_device()
    own = getattr(_ws_local, "ws", None)
    if own is not None and own[0].device.index == key:
        return own
    ws = _ws.get(key)
    if ws is None:
        with _ws_lock:
            ws = _ws.get(key)
            if ws is None:
                ws = (torch.empty(WS_SLAB_BYTES // 4, dtype=torch.float32, device=dev),
                      torch.zeros(WS_COUNTERS, dtype=torch.int32, device=dev))
                _ws[key] = ws
                _all_ws.append(ws)
    return ws


def new_gemm_workspace(dev: torch.device) -> tuple[torch.Tensor, torch.Tensor]:
    """A private split-K workspace (for GEMMs on a second stream)."""
    ws = (torch.empty(WS_SLAB_BYTES // 4, dtype=torch.float32, device=dev),
          torch.zeros(WS_COUNTERS, dtype=torch.int32, device=dev))
    with _ws_lock:
        _all_ws.append(ws)
    return ws


class SplitKFault(RuntimeError):
    """A split-K combine gave up waiting for another slice's partial (gemm_xd / gemm_w4): the
    GEMM that recorded it stored a wrong sum."""


def check_splitk_fault(dev: torch.device | None = None) -> None:
    """Read the fault word (the last counter) of every split-K workspace on ``dev`` (all
    devices: None).  A combine whose poll for the other slices timed out sets it and leaves
    its tile's counters un-armed, so on a fault the counters are zeroed (the next GEMM starts
    clean) and SplitKFault is raised.  Synchronises with the workspace's device: call it after
    warm-up / graph capture and from health checks, not per GEMM."""
    if dev is not None:
        dev = torch.device(dev)
        if dev.type == "cuda" and dev.index is None:
            dev = torch.device("cuda", torch.cuda.current_device())
    with _ws_lock:
        wss = list(_all_ws)
    for slab, cnt in wss:
        if dev is not None and cnt.device != dev:
            continue
        if int(cnt[-1].item()):
            cnt.zero_()
            raise SplitKFault(f"split-K combine timed out on {cnt.device}: a GEMM result since "
                              "the last check is wrong (counters reset)")


class SplitKWatch:
    """Per-step split-K fault detection without a device sync, for one device.

    ``poll()`` (the engine calls it after every step) enqueues, on the current stream, a copy of
    every split-K workspace's fault word into pinned host memory and records an event; a later
    poll reads those words once the event has completed.  A combine that timed out is therefore
    reported one step after the step that ran it (two when the GPU runs a step behind the host),
    instead of up to ``HEALTH_EVERY`` steps later with a blocking read.  On a fault the device's
    counters are zeroed (the next GEMMs start clean) and SplitKFault is raised - or, with
    ``raise_=False``, True is returned."""

    def __init__(self, dev: torch.device):
        dev = torch.device(dev)
        if dev.type == "cuda" and dev.index is None:
            dev = torch.device("cuda", torch.cuda.current_device())
        self.dev = dev
        self._host: torch.Tensor | None = None
        self._ev = None
        self._n = 0

    def _counters(self) -> list[torch.Tensor]:
        with _ws_lock:
            return [cnt for _, cnt in _all_ws if cnt.device == self.dev]

    def poll(self, raise_: bool = True) -> bool:
        if self.dev.type != "cuda":
            return False
        if self._ev is not None and self._ev.query():
            fault = bool(self._host[:self._n].any())
            self._ev = None
            if fault:
                for cnt in self._counters():
                    cnt.zero_()
                if raise_:
                    raise SplitKFault(f"split-K combine timed out on {self.dev}: a GEMM result "
                                      "of the last steps is wrong (counters reset)")
                return True
        if self._ev is None:
            cnts = self._counters()
            if not cnts:
                return False
            if self._host is None or self._host.numel() < len(cnts):
                self._host = torch.zeros(max(4, len(cnts)), dtype=torch.int32, pin_memory=True)
            for i, cnt in enumerate(cnts):
                self._host[i:i + 1].copy_(cnt[-1:], non_blocking=True)
            self._n = len(cnts)
            self._ev = torch.cuda.Event()
            self._ev.record()
        return False


def set_splitk_spin_limit(limit: int) -> int:
    """Bound of the split-K combines' poll for the other slices (polls of ~64 cycles;
    default 1 << 24); < 0 makes every combine fault (tests).  Returns the previous bound."""
    prev = int(hipk().splitk_spin_limit())
    hipk().set_splitk_spin_limit(int(limit))
    return prev


def gemm_w4_variant(variant: int) -> bool:
    """mfma_gemm variants: 7 per-tile (split-K with the last-arriver combine), 9 the same
    with temporal epilogue stores, 11 / 13 per-tile with the parallel split-K combine (every
    slice finishes a row band of its tile; the grid must fit the CUs), 15 persistent, 31
    persistent with the per-XCD K rotation, 47 / 63 those two with the next tile's fragment
    reads spread over half 1."""
    return variant in (7, 9, 11, 13, 15, 31, 47, 63)


def mfma_gemm(x: torch.Tensor, w: torch.Tensor, epi: str = "store",
              residual: torch.Tensor | None = None, out: torch.Tensor | None = None,
              variant: int = 7, splitk: int = 1, group_m: int = 8,
              ws: tuple[torch.Tensor, torch.Tensor] | None = None,
              limit: float = 0.0) -> torch.Tensor:
    """Hand-written CDNA4 GEMM (csrc/kernels/gemm_w4.hip): y = epi(x @ w.T).

    epi "store": y = x @ w.T; "residual": y = x @ w.T + residual (``out`` may be ``residual``
    itself: in-place add into the residual stream); "silu" / "gelu_tanh": w is the fused
    [gate; up] weight [2I, K] and y[:, n] = act(x . gate_n) * (x . up_n) has I columns (no
    act_glu pass); "clamped": the same for the clamped activation bounded by ``limit``; "relu2":
    y = relu(x @ w.T)^2 (both: one K slice, persistent forms or 7).  Shapes: K % 64 == 0,
    N % 256 == 0 (I % 128 == 0 for the gated forms),
    (K / 64) % splitk == 0; rows of x are unrestricted.  ``group_m`` < 0 selects the
    K-slice-by-XCD tile order of the split-K form."""
    assert gemm_w4_variant(variant), variant
    M, K = x.shape
    glu = epi in GATED
    N = w.shape[0] // 2 if glu else w.shape[0]
    if out is None:
        out = torch.empty((M, N), dtype=x.dtype, device=x.device)
    assert out.shape == (M, N) and out.stride(1) == 1, (out.shape, M, N)  # written through ldc
    slab, cnt = ((ws or gemm_workspace(x.device)) if splitk > 1 else (None, None))
    check(hipk().gemm(out.data_ptr(), x.data_ptr(), w.data_ptr(), ptr(residual), M, N, K,
                      x.stride(0), w.stride(0), out.stride(0),
                      residual.stride(0) if residual is not None else 0, EPI[epi],
                      N if glu else 0, variant, splitk, group_m, ptr(slab),
                      slab.numel() * 4 if slab is not None else 0, ptr(cnt),
                      cnt.numel() if cnt is not None else 0, limit, stream_ptr(x)), "gemm")
    return out


def mfma_gemm_grouped(x: torch.Tensor, w: torch.Tensor, grp: torch.Tensor, epi: str = "store",
                      out: torch.Tensor | None = None, group_m: int = 0,
                      ksplit: int = 1, limit: float = 0.0) -> torch.Tensor:
    """Grouped persistent gemm_w4 (csrc/kernels/gemm_w4.hip, V & 64): for every group g,
    out[r] = epi(x[r] @ w[g].T) over the rows r in [grp[g], grp[g + 1]).

    x [R, K] bf16 (rows in group order); w [G, N, K] ("silu" / "gelu_tanh": [G, 2I, K] with
    the gate rows first); grp int32 [G + 1] on the device, non-decreasing, grp[G] <= R -
    read by the kernel, never by the host (a routing kernel writes it: no sync, graph-safe).
    Rows outside [grp[0], grp[G]) of ``out`` are not written.  ``ksplit`` > 1 ("store"): K is
    cut into ksplit slices and out is [ksplit, R, N], slice s holding the bf16 partial product
    over its K range (the consumer sums them; the MoE combine does)."""
    R, K = x.shape
    G_, n2, k2 = w.shape
    glu = epi in GATED
    N = n2 // 2 if glu else n2
    assert k2 == K and w.is_contiguous() and x.stride(1) == 1 and x.dtype == torch.bfloat16
    assert grp.dtype == torch.int32 and grp.numel() == G_ + 1 and grp.device == x.device
    shape = (ksplit, R, N) if ksplit > 1 else (R, N)
    if out is None:
        out = torch.empty(shape, dtype=x.dtype, device=x.device)
    assert out.shape == shape and out.stride(-1) == 1
    if ksplit > 1:
        assert out.is_contiguous()
    check(hipk().gemm_grouped(out.data_ptr(), x.data_ptr(), w.data_ptr(), grp.data_ptr(), G_,
                              R, N, K, x.stride(0), K, out.stride(-2), n2 * K, EPI[epi],
                              N if glu else 0, group_m or (4 if glu else 8), ksplit,
                              R * N if ksplit > 1 else 0, limit, stream_ptr(x)),
          "gemm_grouped")
    return out


def tune(M: int, N: int, K: int, device, iters: int = 20, max_candidates: int = 12) -> dict:
    """Measure every hipBLASLt solution for y[M,N] = x[M,K] @ W[N,K]^T on random operands;
    returns {"algo", "us", "heuristic_us", "candidates"}."""
    g = torch.Generator(device=device).manual_seed(M * 7 + N * 13 + K)
    x = torch.randn(M, K, device=device, dtype=torch.bfloat16, generator=g)
    w = torch.randn(N, K, device=device, dtype=torch.bfloat16, generator=g) * 0.02
    y = torch.empty(M, N, device=device, dtype=torch.bfloat16)
    torch.cuda.synchronize(device)
    res = hipk().lt_tune(y.data_ptr(), x.data_ptr(), w.data_ptr(), M, N, K, K, N, iters,
                         max_candidates, torch.cuda.current_stream(device).cuda_stream)
    if not res:
        raise RuntimeError(f"lt_tune found no solution for M={M} N={N} K={K}")
    heur = next((us for i, us in res if i == -1), float("inf"))
    best_i, best_us = min(((i, us) for i, us in res if i >= 0), key=lambda t: t[1],
                          default=(-1, heur))
    return {"algo": best_i, "us": round(best_us, 2), "heuristic_us": round(heur, 2),
            "candidates": len(res) - 1}


def save_entries(entries: dict[str, dict], path: str | None = None) -> str:
    """Merge ``entries`` ("M,N,K,ldx" -> tune() result) into the table of the running
    hipBLASLt version."""
    path = path or table_path()
    data = load_table(path)
    ver = str(hipk().lt_version())
    cur = data.setdefault(ver, {})
    for k, e in entries.items():
        cur[k] = {**cur.get(k, {}), **e}
    os.makedirs(os.path.dirname(path), exist_ok=True)
    with open(path, "w") as f:
        json.dump(data, f, indent=1, sort_keys=True)
    reset()
    return path


# ------------------------------------------------------------ 4-wave GEMM dispatch
# Persistent gemm_w4 (variant 15: min(tiles, CUs) workgroups, the next tile's first K tiles
# staged during the current tile's last two steps) for every single-slice call.  Against the
# per-tile form in one process (profiles/r3r/probe.log): prefill qkv +0.5 %, o +2.0 %,
# gate_up+GLU +0.9 %, a 4400-row chunk's gate_up+GLU +2.3 %, decode gate_up+GLU at M = 1024
# +4.0 %.  DRTC_W4_PERSIST=0 restores the per-tile form (variant 7).
# Variant 31 (the default) adds the per-XCD K rotation: each XCD label starts its
# K loop at its own eighth of K, so the eight XCDs' epilogue store bursts do not coincide.
# Same box, interleaved (profiles/r4d/seam.log): decode gate_up + GLU at M = 1024 207.4 vs
# 231.1 us (v15), prefill shapes within +-1 % (K = 14336 1.2 % faster).  Fewer than 8 tiles
# run the plain persistent form.
W4_PERSIST = os.environ.get("DRTC_W4_PERSIST", "1") == "1"
# Variant 63 (the default since profiles/r4q) also spreads the next tile's fragment reads
# over half 1 (one per 4 MFMAs after a barrier at MFMA 63, instead of a burst of one per MFMA
# at 104-119): interleaved on one box, prefill gate_up+GLU 2557 vs 2597 us, o+residual 384.9
# vs 392.9, down 1256.6 vs 1280.5, qkv 534.7 vs 531.4, decode gate_up+GLU at M = 1024 199.2
# vs 214.1; headline 20,599 / 20,572 vs 20,338 tok/s.
W4_PERSIST_VARIANT = int(os.environ.get("DRTC_W4_VARIANT", "63"))


def _w4v(K: int) -> int:
    """Schedule variant of a single-slice gemm_w4 call with reduction length K."""
    return W4_PERSIST_VARIANT if W4_PERSIST and K >= 128 else 7


_w4_glu = os.environ.get("DRTC_W4_GLU", "1") != "0"
_w4_plain = os.environ.get("DRTC_W4_GEMM", "1") != "0"
# Prefill-sized passes (M >= W4_MIN_M rows) run the 4-wave hand GEMM (profiles/r3a_w4_gemm.md,
# Llama-3-8B at M = 16384, interleaved with the library in one process):
#   gate_up + SiLU-GLU epilogue  1.03-1.05x hipBLASLt + act_glu   -> hand (no act_glu pass)
#   qkv (store), o (+residual)   0.98-0.99x                        -> hand
#   down (K = 14336, +residual)  0.94-0.96x                        -> library (K > W4_MAX_K)
# gate_up + GLU also wins at the larger decode buckets: 1.04x at M = 768, 1.06x at 1024
# (library + act_glu), 0.97x at 512, 0.72x at 256 (profiles/r3b_w4_decode.md).
W4_GLU_MIN_M = int(os.environ.get("DRTC_W4_GLU_MIN_M", "640"))
W4_MIN_M = int(os.environ.get("DRTC_W4_MIN_M", "4096"))
W4_MAX_K = int(os.environ.get("DRTC_W4_MAX_K", "8192"))


def w4_group_m(M: int, N: int, K: int, glu: bool = False) -> int:
    """Row-tile group of the XCD-aware tile order.  An XCD's 32 workgroups take 32 consecutive
    tiles: with groups of 8 (4) rows that is an 8 x 4 (4 x 8) block of tiles, whose 12 operand
    panels stream through the XCD's L2 per K step, against 18 for the 2 x 16 block of groups
    of 2 (profiles/r5c: hipBLASLt's down kernel 23.4 M L2 misses, gemm_w4 at group 2
    34.1 M).  Interleaved on one box (profiles/r5d): down at K = 14336 1217 us at 8 vs 1247 at
    2; qkv 524 vs 532 at 4; o + residual 376 vs 378; the gated gate_up 2513 at 4 vs 2537 at 8."""
    return 4 if glu else 8


def w4_shape_ok(M: int, N: int, K: int) -> bool:
    """Shapes the prefill-sized hand GEMM takes (tensor strides / alignment aside)."""
    return (_w4_plain and _enabled and M >= W4_MIN_M and K <= W4_MAX_K and K % 64 == 0
            and N % 256 == 0)


def _w4_long(M: int, N: int, K: int) -> bool:
    """Whether gemm_w4 takes a K above W4_MAX_K that no tuned library solution covers.  The library's own
    choice is as good where 256 x 256 tiles come to whole, quarter and three-quarter rounds of the CUs, and
    falls off in between; which, and how far, depends on K and N.  The library's / gemm_w4's time at 4352 ..
    16384 rows, K from 10240, 4096 .. 5120 columns (720 shapes): 0.94 .. 1.76, below 0.98 at six, 1.25 in
    the mean; e.g. 4096 x 11264, 6400 rows 1.44, 8960 1.36, 11520 1.48, 15104 1.29.  Outside: whole and quarter
    rounds there 0.83 .. 1.0, K 8704 and 9216 0.75 .. 1.56 with most below 1, 8192 columns 0.74 .. 1.1 past
    three rounds, 2048 columns 0.84 .. 0.91; K above 16384 below half a round 0.86 .. 1.2."""
    if not (_w4_plain and _enabled and M >= W4_MIN_M and max(10240, W4_MAX_K + 1) <= K <= 28672 and K % 64 == 0
            and N % 256 == 0 and 4096 <= N <= 5120):
        return False
    tiles = -(-M // 256) * (N // 256)
    rounds, part = divmod(tiles, 256)
    even = 256 % (N // 256) == 0  # a round ends with a row of tiles
    if not 384 < tiles < 998 or part == 192:
        return False
    if part >= 128:
        return part < (243 if even and rounds == 2 else 219)
    return K <= 16384 and (0 < part < (51 if even else 38) or part > 76)


def w4_ok(x: torch.Tensor, w: torch.Tensor, residual: torch.Tensor | None = None) -> bool:
    """Whether a prefill-sized projection y = x @ w.T (+ residual) takes gemm_w4."""
    if not _gpu_bf16(x, w):
        return False
    M, K = x.shape
    N = w.shape[0]
    if not (w4_shape_ok(M, N, K) and w.shape[1] == K and _aligned(x, w)):
        return False
    if residual is not None:
        return (residual.dim() == 2 and residual.shape == (M, N) and residual.stride(1) == 1
                and residual.stride(0) % 8 == 0 and residual.data_ptr() % 16 == 0
                and residual.dtype == torch.bfloat16)
    return True


def w4_glu_ok(x: torch.Tensor, w: torch.Tensor, act: str) -> bool:
    """Whether ``norm_glu`` takes the fused-GLU hand GEMM for x [M, K] @ [gate; up]^T."""
    if not (_w4_glu and act in GATED and _gpu_bf16(x, w)):
        return False
    M, K = x.shape
    N2 = w.shape[0]
    return (M >= W4_GLU_MIN_M and K % 64 == 0 and w.shape[1] == K and N2 % 256 == 0
            and _aligned(x, w))


def glu_form(M: int, N2: int, K: int, ldx: int, act: str = "silu") -> int:
    """gemm_xd gated form for a decode batch M through the [gate; up] weight [N2, K]: ``tall_form``'s, or the one the
    tuning table measured fastest (bucket-above for an off-bucket M), else ``_glu_default``, also
    where the table has an entry for the plain product only; 0: none."""
    if not (_xd_enabled and _enabled) or M > DECODE_MAX_M:
        return 0
    tall = tall_form(M, N2 // 2, K, True, act)
    if tall:
        return tall
    found = _decode_entry(M, N2, K, ldx)
    form = found[1][4] if found is not None else 0
    if not form or act == "clamped" and form // 10 % 10 not in XD_CLAMP_NF:
        form = _glu_default(M, N2 // 2, K, act) or _glu_round(M, N2 // 2, K)
    return form if form and xd_supported(M, N2 // 2, K, form, glu=True) else 0


def _glu_round(M: int, I: int, K: int) -> int:
    """gemm_xd gated form of tiles of 256 x 256 that one round takes.  From gemm_w4's first rows where 177 .. 256 of them keep the
    CUs busy, which gemm_w4 takes 2 to 11 % longer for (7168 x 2048 rows of W a half, 1024 rows 56.7 / 53.5 us; 7168 x 4096 99.3 / 89.9;
    6144 x 3072, 800 rows 73.1 / 68.8; 8192 x 4096, 640 95.1 / 86.6; fewer tiles: 5632 x 2048, 896 rows 46.4 / 47.2; more than a
    round: 14336 x 1536 82.3 / 85.4).  Over 2000 sizes K from 1792 on 1.04 .. 1.16, K 1024, 1280 and 1536 0.93, 0.96 and 0.99: gemm_w4's.  From 513 rows where K is short: as fast as the library and a pass on the chip (7168 x
    2048, 560 rows 47.4 / 47.2, 608 47.5 / 49.3), but prompts of these rows, which no decode step is padded to, are as long as their
    host path, and this is one launch for two (two prompts of 300, width 2048: 642 -> 519 a pass)."""
    tiles = -(-M // 256) * (I // 128)
    if tiles > 256 or M > DECODE_MAX_M:
        return 0
    return 281 if M >= W4_GLU_MIN_M and tiles > 176 and K >= 1792 or 512 < M < W4_GLU_MIN_M and K <= 2048 and tiles >= 160 else 0


def _glu_default(M: int, I: int, K: int, act: str = "silu") -> int:
    """gemm_xd gated form of a shape without a measured one, 0 where the library's product and an
    activation pass, or from W4_GLU_MIN_M rows gemm_w4, are as fast.  One launch and no [M, 2 I] intermediate
    win where ``xd_default_form``'s tiles fill the chip: 160 of them, 112 where K is short.  us,
    library + pass / gemm_xd: 7168 x 2048 rows of W a half, 64 rows of x 20.1 / 17.1, 160 29.2 / 20.9, 512
    40.0 / 33.3; 14336 x 4096, 64 rows 59.2 / 48.8; 11008 x 4096, 224 rows 66.5 / 54.0; too few tiles:
    3584 x 4096, 64 rows 21.4 / 24.8.  So do the table's buckets that were tuned without a gated form: 7168 x
    4096, 128 rows 40.9 / 34.6, 448 62.9 / 56.5; 28672 x 8192, 24 rows 169 / 155, 96 199 / 177.
    Tiles of 128 columns a half lose to narrower ones up to 128 rows (28672 x 8192 188 / 199, narrow 179),
    with long K above them (20480 x 8192, 160 rows 179 / 203; 16384 x 4096 154 / 137) and to the library from
    256 rows to gemm_w4's first (14336 x 4096, 320 rows 82 / 97; 7168 x 4096, 600 72 / 87, 5632 x 2048 39 / 48).
    Above 512 rows for the shapes that leave gemm_w4 fewer than three quarters of the CUs: 3584 x 2048, 768 rows
    90 / 29.6, 1024 49 / 30.7; 7168 x 2048, 1024 rows (224 tiles) 53.0 / 53.4.
    The clamped activation has tiles of 64 and 128 columns only: 64 in place of 32 up to 128 rows (7168 x
    2048, 40 rows 20.0 / 18.8, 128 23.7 / 22.1; above, 4096 x 2048, 160 rows 17.3 / 19.3)."""
    if not 17 <= M <= DECODE_MAX_M or M > 512 and -(-M // 256) * (I // 128) > 176:
        return 0
    form = xd_default_form(M, I, K, True)
    if form // 10 % 10 == 8 and M < W4_GLU_MIN_M:
        if M > 256 or M > 128 and K > 4096:
            return 0
        if M <= 128:
            form = 141
    if act == "clamped" and form // 10 % 10 not in XD_CLAMP_NF:
        form = 141 if M <= 128 else 0
    if not form or not xd_supported(M, I, K, form, True):
        return 0
    mt, nf, _ = xd_form(form)
    if -(-M // XD_ROWS[mt]) * (I // (16 * nf)) < (112 if K <= 2048 else 160):
        return 0
    return form + 1000 if xd_nt_ok(M, form) else form


def _stream_glu_ok(x: torch.Tensor, w: torch.Tensor, act: str) -> bool:
    return (act in GATED and _gpu_bf16(x, w) and w.shape[1] == x.shape[1] and w.shape[0] % 2 == 0
            and stream_ok(x.shape[0], w.shape[0] // 2, x.shape[1], act))


def fused_glu_ok(x: torch.Tensor, w: torch.Tensor, act: str) -> bool:
    """Whether ``norm_glu`` computes x [M, K] @ [gate; up]^T with the GLU inside a GEMM
    epilogue (gemm_w4 at prefill-sized / full decode batches, the weight-streaming GEMM at small
    ones, or a tuned gated gemm_xd form)."""
    if w4_glu_ok(x, w, act) or _stream_glu_ok(x, w, act) and _aligned(x, w):
        return True
    return (act in GATED and _gpu_bf16(x, w) and w.shape[1] == x.shape[1] and _staged(x, w)
            and glu_form(x.shape[0], w.shape[0], x.shape[1], x.shape[1], act) != 0)


def norm_glu(p, w: torch.Tensor, act: str = "silu") -> torch.Tensor:
    """h = act(norm(x) @ gate^T) * (norm(x) @ up^T) for an ``ops.PendingNorm`` p and the fused
    [gate; up] weight: on the 4-wave hand GEMM with the GLU in its epilogue when
    ``w4_glu_ok`` (one launch, no [M, 2I] intermediate); at the decode batches where the
    tuner measured it faster, gemm_xd with the GLU in its epilogue; else norm_linear +
    act_glu."""
    from .activation import act_glu

    x = p.x
    if act in ("silu", "gelu_tanh") and isinstance(x, torch.Tensor) and _stream_glu_ok(x, w, act):
        xm = p.materialize()
        if _aligned(xm, w):
            return stream_gemm(xm, w, act)
    if (act in ("silu", "gelu_tanh") and isinstance(x, torch.Tensor) and _gpu_bf16(x, w)
            and w.shape[1] == x.shape[1] and _aligned(x, w)):
        form = glu_form(x.shape[0], w.shape[0], x.shape[1], x.shape[1])  # normed x: dense
        if form:  # a decode batch where the tuner measured the gated gemm_xd fastest
            xm = p.materialize()
            return xd_gemm(xm, w, act, form=form)
    if w4_glu_ok(p.x, w, act):
        x = p.materialize()
        M, K = x.shape
        return mfma_gemm(x, w, act, variant=_w4v(K),
                         group_m=w4_group_m(M, w.shape[0] // 2, K, glu=True))
    return act_glu(norm_linear(p, w), act)


def gated(x: torch.Tensor, w: torch.Tensor, act: str = "silu", limit: float = 0.0) -> torch.Tensor:
    """h = act(x @ gate^T) * (x @ up^T) for normed rows x and the fused [gate; up] weight, by
    the same choice of kernels as ``norm_glu``; ``limit``: bound of the clamped activation."""
    from .activation import act_glu

    if _stream_glu_ok(x, w, act) and _aligned(x, w):
        return stream_gemm(x, w, act, limit=limit)
    if fused_glu_ok(x, w, act):
        M, K = x.shape
        form = glu_form(M, w.shape[0], K, x.stride(0), act)
        if form:
            return xd_gemm(x, w, act, form=form, limit=limit)
        return mfma_gemm(x, w, act, variant=_w4v(K), limit=limit,
                         group_m=w4_group_m(M, w.shape[0] // 2, K, glu=True))
    return act_glu(linear(x, w), act, limit=limit)


def squared_relu(x: torch.Tensor, w: torch.Tensor, out: torch.Tensor) -> torch.Tensor:
    """out = relu(x @ w.T)^2, into rows of any stride (columns of a wider operand): in the
    epilogue of gemm_w4 at prefill size and of gemm_xd or the weight-streaming GEMM where ``linear``
    takes those, else a pass behind ``linear``."""
    M, K = x.shape
    assert out.shape == (M, w.shape[0]) and out.stride(1) == 1
    if not on_gpu(x):
        out.copy_(F.relu(F.linear(x, w)).square())
        return out
    if w4_ok(x, w) and out.stride(0) % 8 == 0 and out.data_ptr() % 16 == 0:
        return mfma_gemm(x, w, "relu2", out=out, variant=_w4v(K),
                         group_m=w4_group_m(M, w.shape[0], K))
    if _gpu_bf16(x, w) and w.shape[1] == K and _aligned(x, w) and out.stride(0) % 8 == 0 and out.data_ptr() % 16 == 0:
        kind, form = route(M, w.shape[0], K, x.stride(0))
        if (kind, form) == ("skinny", STREAM):
            return stream_gemm(x, w, "relu2", out=out)
        if kind == "xd" and _staged(x, w):
            return xd_gemm(x, w, "relu2", out=out, form=form)
        if kind == "skinny" and out.dtype == x.dtype:
            N = w.shape[0]
            check(hipk().skinny_gemm(out.data_ptr(), x.data_ptr(), w.data_ptr(), M, N, K, x.stride(0), out.stride(0), form,
                                     0, 0, 0, 0, 0, 0, 1, stream_ptr(x)), "skinny_gemm")
            return out
    y = linear(x, w)
    check(hipk().relu2(int(y.dtype == torch.float32), out.data_ptr(), out.stride(0), y.data_ptr(),
                       M, w.shape[0], stream_ptr(x)), "relu2")
    return out


# ------------------------------------------------------------------ XCD-partitioned decode GEMM
XD_EPI = {"store": 0, "residual": 1, "silu": 2, "gelu_tanh": 3, "clamped": 4, "relu2": 5}
# tile shapes built in gemm_xd.hip, (mt, nf) -> LDS ring depth (XD_ROWS[mt] x 32 nf tiles); a form
# is mt * 100 + nf * 10 + splitk (K split over 1..8 slices), + 1000 for non-temporal weight
# loads (the tiles of XD_NT_TILES)
XD_TILES = {(0, 1): 6, (0, 2): 6, (0, 4): 4, (3, 2): 5, (3, 4): 4, (4, 4): 4, (5, 4): 3, (1, 2): 4, (1, 4): 4, (1, 6): 3, (2, 4): 3, (2, 6): 2, (2, 8): 2}
XD_ROWS = {0: 64, 1: 128, 2: 256, 3: 160, 4: 192, 5: 224}  # mt -> rows of a tile
XD_CLAMP_NF = (4, 8)  # tile widths the clamped epilogue is built for
XD_NT_TILES = {(0, 1), (0, 2), (0, 4), (3, 2), (3, 4), (4, 4), (5, 4), (1, 4), (1, 6), (2, 4), (2, 6), (2, 8)}
XD_MAX_SPLITK = 8
# the forms the tuner (scripts/tune_xd.py) measures
XD_FORMS = tuple(sorted([mt * 100 + nf * 10 + 1 for mt, nf in XD_TILES if 1 <= mt <= 2] +
                        [200 + nf * 10 + sk for nf in (4, 6, 8) for sk in (2, 3, 4)]))


def xd_form(form: int) -> tuple[int, int, int]:
    return form % 1000 // 100, form // 10 % 10, form % 10


def xd_nt(form: int) -> bool:
    """Form with non-temporal weight loads."""
    return form >= 1000


@functools.lru_cache(maxsize=4096)  # (asked several times a layer; of its arguments alone)
def xd_supported(M: int, N: int, K: int, form: int, glu: bool = False) -> bool:
    """Shapes gemm_xd.hip takes in ``form`` (mt * 100 + nf * 10 + splitk); N = output
    columns (gated: half the rows of the [gate; up] weight)."""
    mt, nf, sk = xd_form(form)
    if (mt, nf) not in XD_TILES or not 1 <= sk <= XD_MAX_SPLITK or (glu and nf % 2) or mt == 0 and (glu or sk > 1):
        return False
    if mt > 2 and not (xd_nt(form) and sk == 1 and M <= XD_ROWS[mt]):  # one row tile, non-temporal
        return False
    if form // 1000 > 1 or (xd_nt(form) and (mt, nf) not in XD_NT_TILES):
        return False
    tno = 16 * nf if glu else 32 * nf
    if not (M >= 1 and N % tno == 0 and K % 64 == 0 and K // 64 // sk > XD_TILES[(mt, nf)]):
        return False
    # split-K: the partial slots and tile counters fit the device workspace
    rows = XD_ROWS[mt]
    tiles = -(-M // rows) * (N // tno)
    return sk == 1 or (tiles * sk * rows * (32 * nf) * 4 <= WS_SLAB_BYTES
                       and 2 * tiles + 2 <= WS_COUNTERS)  # + the fault word (last counter)


@functools.lru_cache(maxsize=4096)
def xd_default_form(M: int, N: int, K: int, glu: bool = False) -> int:
    """Form of an untuned shape, by a per-CU operand-bytes model (profiles/r4i): a CU's
    time ~ (tile rows + columns) x (K / splitk) x 2 B per round of 256 work items, plus the
    split-K combine (its fp32 partials, weighted 5x: measured far costlier than their bytes)."""
    best, cost = 0, None
    for form in XD_FORMS:
        if not xd_supported(M, N, K, form, glu):
            continue
        mt, nf, sk = xd_form(form)
        tno, rows = 16 * nf if glu else 32 * nf, XD_ROWS[mt]
        items = -(-M // rows) * (N // tno) * sk
        rounds = -(-items // 256)
        c = rounds * ((rows + 32 * nf) * (K // sk) * 2 + 100_000
                      + 5 * (sk - 1) * rows * (32 * nf) * 4)
        if cost is None or c < cost:
            best, cost = form, c
    return best


def xd_gemm(x: torch.Tensor, w: torch.Tensor, epi: str = "store",
            residual: torch.Tensor | None = None, out: torch.Tensor | None = None,
            form: int = 0, ws: tuple[torch.Tensor, torch.Tensor] | None = None,
            limit: float = 0.0) -> torch.Tensor:
    """Decode-shaped hand GEMM, csrc/kernels/gemm_xd.hip: y = epi(x @ w.T) on tiles of XD_ROWS[mt] rows x 32 nf
    columns, K split over 1..8 slices, with the tile order partitioned by XCD (each XCD streams
    its own weight column panels through its L2 for every row tile).  mt 0 (64 rows): plain, one slice; mt 3 to 5 (160, 192
    and 224 rows): one row tile, one slice, non-temporal weight loads.  epi "store";
    "residual" (``out`` may be ``residual``); "silu" / "gelu_tanh": w is the fused [gate; up]
    weight [2I, K] and y[:, n] = act(x . gate_n) * (x . up_n); "clamped": bounded by ``limit``
    (tiles of XD_CLAMP_NF); "relu2": relu(x @ w.T)^2.  ``form`` = mt * 100 + nf * 10 + splitk (+ 1000: non-temporal weight loads; 0: ``xd_default_form``)."""
    M, K = x.shape
    glu = epi in GATED
    N = w.shape[0] // 2 if glu else w.shape[0]
    form = form or xd_default_form(M, N, K, glu)
    assert xd_supported(M, N, K, form, glu), (M, N, K, form, epi)
    assert x.dtype == w.dtype == torch.bfloat16 and x.stride(1) == 1 and w.is_contiguous()
    mt, nf, sk = xd_form(form)
    if out is None:
        out = residual if (epi == "residual" and residual is not None) else \
            torch.empty((M, N), dtype=x.dtype, device=x.device)
    # the kernel writes M x N through ldc: the output must hold exactly that
    assert out.shape == (M, N) and out.stride(1) == 1 and out.dtype == x.dtype, (out.shape, M, N)
    if epi == "residual":
        assert residual is not None and residual.shape == (M, N) and residual.stride(1) == 1
    slab, cnt = ((ws or gemm_workspace(x.device)) if sk > 1 else (None, None))
    check(hipk().gemm_xd(out.data_ptr(), x.data_ptr(), w.data_ptr(), ptr(residual), M, N, K,
                         x.stride(0), w.stride(0), out.stride(0),
                         residual.stride(0) if residual is not None else 0, XD_EPI[epi],
                         mt | (16 if xd_nt(form) else 0), nf,
                         sk, ptr(slab), slab.numel() * 4 if slab is not None else 0, ptr(cnt),
                         cnt.numel() if cnt is not None else 0, limit, stream_ptr(x)), "gemm_xd")
    return out


# ------------------------------------------------------------------ medium-M decode GEMM
MIDM_EPI = {"store": 0, "residual": 1, "silu": 2, "gelu_tanh": 3}  # 4: partial sums (``linear_parts``)
MIDM_MAX_M = 256


def midm_splits(M: int, N: int, K: int, target_wgs: int = 256) -> int:
    """K splits of the medium-M GEMM: the largest S <= 16 with K a multiple of 256 S and at most one workgroup per
    CU, since its ring takes the whole LDS (us, two / one: 4096 x 4096, 24 rows 17.0 / 12.6; 4096 x 14336, 64 rows 36.5 /
    28.7; 8192 x 28672, 64 rows 94.9 / 82.7)."""
    nb = N // 128
    ring = 64 * midm_depth(M)
    best = 1
    for s in range(1, 17):
        if K % (ring * s) == 0 and nb * s <= target_wgs:
            best = s
    return best


def midm_depth(M: int) -> int:
    """K tiles of 64 that a split of ``midm_splits`` is a multiple of."""
    return 4


def midm_supported(M: int, N: int, K: int, epi: str = "store") -> bool:
    return (1 <= M <= MIDM_MAX_M and N % 128 == 0 and K % 64 == 0
            and epi in MIDM_EPI
            and (epi not in ("silu", "gelu_tanh") or (N // 2) % 4 == 0))


def midm_gemm(x: torch.Tensor, w: torch.Tensor, epi: str = "store",
              residual: torch.Tensor | None = None, out: torch.Tensor | None = None,
              splits: int | None = None, nf: int = 4) -> torch.Tensor:
    """Medium-M (up to 256 rows) decode GEMM, csrc/kernels/gemm_midm.hip: y = x @ w^T with a
    store / residual (y = residual + x w^T, in place when out is residual) / SiLU- or
    GELU-gated [gate | up] epilogue.  Tiles of all rows and 32 ``nf`` (2, 4) columns, K split over
    workgroups, the fp32 partials summed by a second small kernel."""
    M, K = x.shape
    N = w.shape[0]
    assert x.dtype == torch.bfloat16 and w.dtype == torch.bfloat16 and x.is_cuda
    assert x.stride(1) == 1 and w.is_contiguous() and w.shape[1] == K
    assert midm_supported(M, N, K, epi) or nf == 2 and N % 64 == 0 and midm_supported(M, 2 * N, K, epi), (M, N, K, epi)
    S = splits or midm_splits(M, N, K)
    while S > 1 and S * M * N * 4 > WS_SLAB_BYTES:
        S //= 2
    NO = N // 2 if epi in ("silu", "gelu_tanh") else N
    if out is None:
        out = residual if (epi == "residual" and residual is not None) else \
            torch.empty((M, NO), dtype=x.dtype, device=x.device)
    assert out.shape == (M, NO) and out.stride(1) == 1
    if epi == "residual":
        assert residual is not None and residual.shape == (M, N) and residual.stride(1) == 1
    # whole 16-byte pieces into LDS at 32-bit offsets, residual and y by four values: what lies otherwise is copied
    if x.stride(0) % 8 == 0 and (x.data_ptr() % 16 or x.stride(0) >= 1 << 22):
        x = torch.empty((M, K), dtype=x.dtype, device=x.device).copy_(x)
    if w.data_ptr() % 16:
        w = w.clone()
    if residual is not None and residual.stride(0) % 4 == 0 and residual.data_ptr() % 8:
        residual = torch.empty((M, N), dtype=x.dtype, device=x.device).copy_(residual)
    if out.stride(0) % 4 == 0 and out.data_ptr() % 8:
        return out.copy_(midm_gemm(x, w, epi, residual, torch.empty((M, NO), dtype=x.dtype, device=x.device), splits, nf))
    slab = gemm_workspace(x.device)[0]
    check(hipk().midm_gemm(out.data_ptr(), x.data_ptr(), w.data_ptr(), ptr(residual), M, N, K,
                           x.stride(0), out.stride(0),
                           residual.stride(0) if residual is not None else 0, MIDM_EPI[epi], S, nf,
                           slab.data_ptr(), slab.numel() * 4, stream_ptr(x)), "midm_gemm")
    return out


class Parts:
    """x @ w.T as the fp32 sums of its K slices, ``slab`` [S, M, N], for an op that adds them up while it
    reads its input (``PendingNorm`` with a residual, ``dyt``, ``fused_moe``'s ``y``)."""

    __slots__ = ("slab", "dtype")

    def __init__(self, slab: torch.Tensor, dtype: torch.dtype):
        self.slab, self.dtype = slab, dtype

    @property
    def shape(self) -> torch.Size:
        return self.slab.shape[1:]

    def tensor(self) -> torch.Tensor:
        return self.slab.sum(0).to(self.dtype)


MAX_PARTS = 8  # common.h kMaxParts
_parts_enabled = os.environ.get("DRTC_PARTS", "1") != "0"
# (M, N, K, most) -> (16-column fragments, K slices) of ``linear_parts``, None: ``linear``
_parts_forms: dict[tuple[int, int, int, int], tuple[int, int] | None] = {}


def parts_form(M: int, N: int, K: int, most: int = MAX_PARTS) -> tuple[int, int] | None:
    """How ``linear_parts`` cuts a product of M rows into up to ``most`` slices, None where ``linear`` is as fast.  us of
    ``linear`` as it was before ``small_form`` / of the parts, to which reading them adds 0.3 - 2:
      K from 5120 on, 3 rows to 256: 4096 x 14336, 4 rows 22.7 / 19.8, 16 24.2 / 19.8, 64 28.3 / 22.7, 160 39.0 / 30.8, 256
        58.0 / 38.6; 2048 x 7168, 4 rows 11.0 / 7.4, 160 24.2 / 14.1; 2048 x 5632, 256 rows 20.9 / 16.0; two rows and one
        stay with the dot2 form (2048 x 7168 8.4 / 7.4, 7.5 / 7.3)
      K from 4096 on to 160 rows: 4096 x 4096, 4 rows 9.7 / 8.4, 16 11.1 / 8.5, 64 14.1 / 9.9, 160 19.5 / 15.0; 200 18.8 / 17.3
      K from 2048 on, 17 rows to 64, 128 where narrow: 2048 x 2048, 16 rows 6.2 / 4.8, 24 7.6 / 5.0, 64 10.7 / 5.9, 128 10.7 /
        7.6, 160 10.5 / 8.7; 3584 x 2048, 64 rows 9.4 / 7.0, 96 9.2 / 8.3
    Product and norm together, ``linear`` as it is / the parts: over 1224 shapes of K 2048 to 28672 1 / 0.72; 4096 x 14336,
      4 rows 27.2 / 25.6, 64 31.1 / 29.6, 256 52.1 / 49.3; 2048 x 7168, 160 rows 26.7 / 20.7; 4096 x 4096, 16 rows 14.2 / 12.5, 64
      17.2 / 14.9; 2048 x 2048, 24 rows 9.7 / 8.0, 64 10.8 / 9.3.  The 64-row tiles of ``small_form`` are the faster product in
      52 of them, most of K up to 4096 from 96 rows on (4096 x 4096, 144 rows 20.2 / 23.8; 2048 x 2048, 128 rows 10.9 / 12.6),
      and for 256 rows at K near 5120 (1024 x 5120 17.0 / 19.7).  The parts stay there: the norm reads these sums in 32 bits,
      and a product's rows would be rounded to 16 in between.
    The cut: the least of a workgroup's operands at 50 GB/s or its weights at 24, a quarter of a microsecond to
    a slice, and the parts read again by the whole chip or by a row's CU."""
    key = (M, N, K, most)
    if key in _parts_forms:
        return _parts_forms[key]
    rows = (3, 256) if K >= 5120 else (3, 160) if K >= 4096 else (17, 128 if N <= 2048 else 64) if K >= 2048 else (1, 0)
    best = None
    if _parts_enabled and _midm_enabled and K % 64 == 0 and 1024 <= N <= 8192 and rows[0] <= M <= rows[1]:
        for nf in (2, 4):
            for s in range(2, most + 1):
                tiles = N // (32 * nf) * s
                if N % (32 * nf) or tiles > 256 or K // 64 // s < 4:
                    continue
                cost = (max(K / s * (M + 32 * nf) * 2 / 50e3, K / s * 32 * nf * 2 / 24e3) + 0.25 * s
                        + max(s * M * N * 4 / 8e6, s * N * 4 / 65e3))
                if best is None or cost < best[0]:
                    best = cost, (nf, s)
    form = best[1] if best else None
    _parts_forms[key] = form
    return form


def linear_parts(x: torch.Tensor, w: torch.Tensor, most: int = MAX_PARTS) -> torch.Tensor | Parts:
    """``linear``, or the sums of up to ``most`` K slices (csrc/kernels/gemm_midm.hip) where ``parts_form`` says so."""
    if x.shape[0] > MIDM_MAX_M:  # (a prompt's host path is as long as its kernels up to some 600 rows)
        return linear(x, w)
    if _gpu_bf16(x, w) and w.shape[1] == x.shape[1] and _aligned(x, w):
        (M, K), N = x.shape, w.shape[0]
        form = parts_form(M, N, K, most) if M * x.stride(0) < 1 << 30 else None
        if form is not None:
            nf, S = form
            slab = torch.empty((S, M, N), dtype=torch.float32, device=x.device)
            check(hipk().midm_gemm(0, x.data_ptr(), w.data_ptr(), 0, M, N, K, x.stride(0), N, 0, 4, S, nf,
                                   slab.data_ptr(), slab.numel() * 4, stream_ptr(x)), "midm_gemm")
            return Parts(slab, x.dtype)
    return linear(x, w)


__all__ = ["linear", "linear_beside", "linear_parts", "parts_form", "Parts", "route", "norm_linear", "glu_linear", "norm_glu_row", "norm_glu", "fused_glu_ok",
           "linear_residual",
           "residual_fusable", "w4_glu_ok", "w4_ok", "w4_shape_ok", "squared_relu", "w4_group_m", "mfma_gemm",
           "mfma_gemm_grouped",
           "gemm_workspace", "new_gemm_workspace", "private_workspace", "check_splitk_fault", "SplitKFault", "SplitKWatch",
           "set_splitk_spin_limit", "skinny_linear", "skinny_ok",
           "skinny_variant", "skinny_supports", "midm_gemm", "midm_supported", "midm_splits",
           "stream_gemm", "stream_ok", "stream_slices", "xd_gemm", "xd_supported", "xd_default_form", "tune", "save_entries", "load_table", "reset", "set_enabled", "table_path"]
