"""Linear layers on hand-written MFMA kernels, autotuned per decode bucket, with fused epilogues.

``linear(x, w)`` computes ``x @ w.T`` (w stored [N, K], K contiguous).
``linear_swiglu(gu, w)`` computes ``silu(gu[:, :K]) * gu[:, K:] @ w.T``.

Kernels (csrc/kernels):
  * ``tgemm.hip``  — LDS-tiled MFMA GEMM (global_load_lds ring, XOR-swizzled LDS, XCD-aware
    block order, optional in-launch split-K) with the transformer epilogues used by the fused
    decoder layer (models/llama.py): QKV + RoPE + paged-KV write, residual add + row sums of
    squares (RMSNorm folded into the next GEMM), SwiGLU.  Any M (decode buckets and prefill).
  * ``decode_gemm.hip`` (M <= 64): decode GEMMs with the same epilogues on fragment-major weight copies (``frag_weight``).
  * ``gemv.hip`` (M <= 8), ``skinny_gemm.hip`` (M <= 128): register-streaming decode GEMMs without
    LDS tiling, on row-major weights.
  * hipBLASLt via ``F.linear`` stays a candidate, so a custom kernel is used only where it wins.

Plans are measured once per (M, N, K) OUTSIDE graph capture (``autotune``, called by the engine
for every decode bucket before capturing) as hipGraph replays over rotated weight copies (a
decode step streams the whole model: weights come from HBM, not the Infinity Cache); an unseen
shape (prefill) uses a heuristic plan.  CPU tensors -> plain torch.

Split-K workspaces are FIXED-size per (device, owner) and never re-allocated: captured graphs
keep raw pointers to them, so growing (freeing) a workspace after a capture would leave graph
replays writing into freed memory.  Plans whose workspace need exceeds the fixed
size are never chosen.  Engines capture under their own owner key (``workspace_owner``), so two
engines replaying graphs concurrently on one device never share split-K tickets.
"""
from __future__ import annotations

import contextlib
import contextvars
import json
import math
import os
from typing import Dict, Iterable, List, Optional, Tuple

import torch
import torch.nn.functional as F

from . import _load as _load_ext, _native, reference as ref

MAX_M = 1024       # decode buckets up to this size are autotuned
SKINNY_MAX_M = 128
_SPLITS = (1, 2, 4, 8, 16)
_NTWS = (1, 2, 4)
_GEMV_MS = (1, 2, 4, 8)   # csrc/kernels/gemv.hip instantiations (decode buckets below 16)
SKE_MAX_M = 16            # small-batch MFMA GEMM with fused epilogues (skinny_gemm.hip skinny_epi_kernel)
_SKE_SPLITS = (1, 2, 4, 8)
_GEMV_RS = (1, 2, 4)
_TG_TILES = ((64, 64, 4), (64, 128, 4), (128, 64, 4), (128, 128, 4), (64, 128, 8), (128, 128, 8), (192, 128, 8),
             (256, 128, 8),
             (256, 256, 8))
_TG_SPLITS = (1, 2, 3, 4, 6, 8)
# loader-wave plans (csrc/kernels/tgemm.hip by_tile_nl): (bm, bn, compute waves, stages, loader waves);
# M is the smallest batch each is tried at (larger tiles only pay once M fills them)
# (8 loader waves: a CU's LDS-DMA intake grows with the waves issuing it, ~75 GB/s at 4 and ~140 GB/s
# at 8 on contiguous pieces, scripts/exp/intake.hip; profiles/r3_decode_gemm_panel.md)
_TG_NL = ((16, 128, 4, 4, 6, 1), (16, 128, 4, 8, 6, 1),   # batch <= 16 only (TG_NL16_MAX_M): 16-row tiles
          (64, 64, 4, 4, 4, 1), (128, 64, 4, 4, 4, 65), (160, 128, 8, 3, 4, 129), (256, 128, 8, 3, 4, 129),
          (64, 64, 4, 4, 8, 1), (64, 64, 4, 8, 8, 1), (128, 64, 4, 4, 8, 65), (128, 128, 4, 4, 8, 65),
          (160, 128, 8, 3, 6, 129), (256, 128, 8, 3, 8, 129))
# 32-deep k-step plans (csrc/kernels/tgemm.hip by_tile_k32): (bm, bn, stages, loaders), 8 compute waves;
# as plan tuples (bm, bn, stages, splits, 1, 8, 1, loaders, 0, 32)
_TG_K32 = ((256, 256, 4, 0),)
# 32 x 32 x 16 MFMA plans (csrc/kernels/tgemm.hip by_tile_m32), as full plan tuples with k depth 64 and
# mfma 32: the flagship's 64-row decode tiles, measured against everything else (the 128- and 256-row
# forms lost 6-16 % to 16 x 16 x 32 and are pruned: profiles/r6_gemm_fill_path.md, r6_prune.md)
_TG_M32 = ((64, 64, 3, 1, 2, 4, 1, 0, 0, 64, 32), (64, 128, 3, 1, 2, 8, 1, 0, 0, 64, 32))
# plans no measured shape ever selected, not instantiated (csrc/kernels/tgemm.hip kPruned, same table):
# (bm, bn, stages, ks, waves, wk, loaders, k depth, mfma); profiles/r6_prune.md
_TG_PRUNED = frozenset({
    (64, 128, 6, 1, 4, 1, 0, 64, 16), (64, 128, 2, 2, 4, 1, 0, 64, 16), (128, 64, 3, 1, 4, 1, 0, 64, 16),
    (128, 64, 4, 1, 4, 1, 0, 64, 16), (128, 64, 6, 1, 4, 1, 0, 64, 16), (128, 64, 2, 2, 4, 1, 0, 64, 16),
    (128, 64, 3, 2, 4, 1, 0, 64, 16), (128, 128, 3, 1, 4, 1, 0, 64, 16), (128, 128, 4, 1, 4, 1, 0, 64, 16),
    (128, 128, 2, 2, 4, 1, 0, 64, 16), (64, 128, 2, 1, 8, 1, 0, 64, 16), (64, 128, 2, 2, 8, 1, 0, 64, 16),
    (128, 128, 2, 1, 8, 1, 0, 64, 16), (128, 128, 2, 2, 8, 1, 0, 64, 16), (192, 128, 2, 1, 8, 1, 0, 64, 16),
    (256, 128, 2, 1, 8, 1, 0, 64, 16), (64, 128, 2, 2, 4, 2, 0, 64, 16),
    (128, 64, 2, 2, 4, 2, 0, 64, 16), (128, 64, 3, 2, 4, 2, 0, 64, 16), (128, 128, 2, 2, 4, 2, 0, 64, 16),
    (64, 64, 4, 1, 4, 1, 2, 64, 16), (64, 64, 8, 1, 4, 1, 4, 64, 16), (128, 128, 4, 1, 4, 1, 4, 64, 16),
    (256, 128, 6, 1, 8, 1, 0, 32, 16), (256, 128, 6, 1, 8, 1, 8, 32, 16), (128, 64, 4, 1, 4, 1, 8, 64, 32),
    (256, 128, 3, 1, 8, 1, 8, 64, 32), (256, 256, 2, 1, 8, 1, 0, 64, 32),
})


def tg_built(plan) -> bool:
    """False for a plan tuple (bm, bn, stages, splits, ks, waves[, wk, loaders, sk, k depth, mfma, raster])
    whose kernel is pruned from the build."""
    p = tuple(plan) + (1, 0, 0, 64, 16)[max(0, len(plan) - 6):]
    return (p[0], p[1], p[2], p[4], p[5], p[6], p[7], p[9], p[10]) not in _TG_PRUNED


# one-split plans with a stream-K instantiation (csrc/kernels/tgemm.hip sk_plan, PLAIN epilogue only):
# (bm, bn, stages, ks, waves, loaders)
_SK_PLANS = {(64, 64, 3, 2, 4, 0), (64, 64, 4, 1, 4, 0), (64, 64, 4, 1, 4, 4), (64, 64, 4, 1, 4, 8),
             (64, 128, 3, 1, 8, 0), (128, 64, 4, 1, 4, 4)}
WS_FLOATS = 16 << 20      # 64 MiB of f32 split-K slabs per (device, owner)
WS_COUNTERS = 1 << 16

EPI_PLAIN, EPI_RESADD, EPI_QKV, EPI_SWIGLU, EPI_GELU = 0, 1, 2, 3, 4
DG_GLU, DG_GELU = 4, 5      # of the decode GEMM alone

# K-panel-major weight copies for the fused decoder GEMMs (GemmArgs.w_panel): every tgemm ring fill
# of the weight operand is one contiguous 1 KB instead of eight 128-B row pieces 4-11 KB apart
# (profiles/r3_decode_gemm_panel.md).  The row-major weight stays for the GEMV / skinny / hipBLASLt
# paths; models.llama keeps the panel copy only while both fit comfortably in HBM.
W_PANEL = True


def panel_weight(w: torch.Tensor) -> torch.Tensor:
    """[N, K] -> [K / 64, N, 64] (element (n, k) at ((k // 64) N + n) 64 + k % 64)."""
    N, K = w.shape
    return w.view(N, K // 64, 64).transpose(0, 1).contiguous()


def copies_fit(extra: int, device, spare: int = 0) -> bool:
    """May a model lay out ``extra`` bytes of further weight copies?  While they fit in a quarter of the device memory still free beyond
    ``spare`` bytes (e.g. not Llama-3-70B at TP=1: 141 GB of weights on a 288 GB part; co-located engines and processes sharing the GPU
    each see what the others left), and never in the one-GPU multi-rank rehearsal (N processes would each add a copy on one card)."""
    return os.environ.get("DLLM_REHEARSE_ONE_GPU") != "1" and extra <= 0.25 * (torch.cuda.mem_get_info(device)[0] - spare)


# Fragment-major weight copies of the decode GEMM (csrc/kernels/decode_gemm.hip): a wave's load of a weight fragment is one contiguous
# 1 KB instead of 16 rows of 64 bytes.
DG_MAX_M = 64
_PAIR_ROWS = [*range(8), *range(16, 24), *range(8, 16), *range(24, 32)]


def frag_weight(w: torch.Tensor, paired=False) -> torch.Tensor:
    """[N, K] -> [ceil(N / 16), K / 32, 64, 8]: of a 16-column tile and 32 k, lane 16 g + r holds W[16 t + r][32 s + 8 g ...+ 7]; rows past
    N are zeros.  ``paired`` (the QKV and gate|up weights of models.llama, pairs 16 rows apart in groups of 32): pairs 8 rows apart; "glu": gate rows, then up rows, likewise.
    f32: [ceil(N / 16), K / 16, 64, 4], lane 16 g + r holds W[16 t + r][16 s + 4 g ...+ 3] (f32_gemm)."""
    N, K = w.shape
    if w.dtype == torch.float32:
        if K % 16 or paired:
            raise ValueError(f"frag_weight: {N} x {K}")
        w = torch.cat([w, w.new_zeros(-N % 16, K)])
        return w.view(-1, 16, K // 16, 4, 4).permute(0, 2, 3, 1, 4).reshape(-1, K // 16, 64, 4).contiguous()
    if paired == "glu":
        if K % 32 or N % 16:
            raise ValueError(f"frag_weight: {N} x {K}")
        return frag_weight(w.view(2, N // 16, 8, K).transpose(0, 1).reshape(N, K))
    if K % 32 or (paired and N % 32):
        raise ValueError(f"frag_weight: {N} x {K}")
    if paired:
        w = w.view(N // 32, 32, K)[:, _PAIR_ROWS].reshape(N, K)
    elif N % 16:
        w = torch.cat([w, w.new_zeros(16 - N % 16, K)])
    return w.view(-1, 16, K // 32, 4, 8).permute(0, 2, 3, 1, 4).reshape(-1, K // 32, 64, 8).contiguous()


def _nk(w: torch.Tensor) -> Tuple[int, int]:
    """(N, K) of a row-major [N, K] or panel [K / 64, N, 64] weight."""
    return (w.shape[1], w.shape[0] * 64) if w.dim() == 3 else (w.shape[0], w.shape[1])

_OWNER: contextvars.ContextVar = contextvars.ContextVar("dllm_gemm_ws_owner", default=None)


@contextlib.contextmanager
def workspace_owner(key):
    """Route split-K workspace lookups of this thread/context to ``key``'s own buffers."""
    tok = _OWNER.set(key)
    try:
        yield
    finally:
        _OWNER.reset(tok)


class _Planner:
    def __init__(self):
        self.plans: Dict[Tuple[int, int, int, bool], Tuple] = {}     # best overall, for linear()
        self.tg_plans: Dict[Tuple[int, int, int], Tuple] = {}        # best tgemm tile, for the fused ops
        # decode GEMM (nt, vs, splits) where it beats plans[...], None where it was timed and does not
        self.dg_plans: Dict[Tuple[int, int, int], Optional[Tuple]] = {}
        self.fused_core: Dict[Tuple[int, int, int], str] = {}        # "tg" | "lin" | "gemvR" | "skES" per tuned shape
        # the same with "dgN.V.S" among the choices, for weights that have fragment-major copies: whether a model has them is decided by
        # the memory that is free when it is made, so both kinds may run in one process or load one plan file
        self.frag_core: Dict[Tuple[int, int, int], str] = {}
        self.fused_opts: Dict[Tuple[int, int, int], Dict[str, float]] = {}   # measured us per core choice
        self.pf_times: Dict[Tuple[int, int], list] = {}      # (N, K) of prompts: [(plan, rows, us)]
        self.pf_small: Dict[Tuple[int, int, int], Tuple] = {}        # (rows of PF_SMALL_MS, N, K): (fastest plan, its us)
        self.pf_tail: Dict[Tuple[int, int, int], Tuple] = {}        # the same of PF_TAIL_MS
        self.pf_lin: Dict[Tuple[int, int], list] = {}        # (N, K) of prompts: [(rows, us)] of the vendor's product and its epilogue
        self.pf_parts: Dict[Tuple[int, int, int], Tuple] = {}        # prompt_parts' answers
        self.pf_vendor: Dict[Tuple[int, int, int], bool] = {}        # use_vendor_core's, for rows that are no bucket
        # (N, K, 1 with a GELU behind it) of plain products of prompts: [(rows, us of the vendor's, GELU's launch included)], [(rows, us of
        # each of _PP_PLANS)]
        self.pp_times: Dict[Tuple[int, int, int], Tuple[list, list]] = {}
        self.pp_plans: Dict[Tuple[int, int, int, int], Optional[Tuple]] = {}      # prompt_plan's answers
        self.cus = 256            # CUs of the device the prompt plans were timed on
        self.ws: Dict[Tuple, Tuple[torch.Tensor, torch.Tensor]] = {}
        self.sk_tables: Dict[Tuple, Tuple[torch.Tensor, int]] = {}   # stream-K segment lists per shape
        self.timings: Dict[Tuple[int, int, int, bool], Dict[str, float]] = {}

    def workspace(self, dev: torch.device, floats: int, tiles: int):
        """The fixed (part, counters) pair of the current owner on ``dev``; created once, outside
        capture, never grown."""
        if floats > WS_FLOATS or tiles > WS_COUNTERS:
            raise RuntimeError(f"split-K plan needs {floats} floats / {tiles} tickets > fixed workspace")
        key = (str(dev), _OWNER.get())
        w = self.ws.get(key)
        if w is None:
            if torch.cuda.is_current_stream_capturing():
                raise RuntimeError("split-K workspace first touched during graph capture (call reserve())")
            w = (torch.empty(WS_FLOATS, dtype=torch.float32, device=dev),
                 torch.zeros(WS_COUNTERS, dtype=torch.int32, device=dev))
            self.ws[key] = w
        return w


_P = _Planner()


def reserve(device) -> None:
    """Create the current owner's workspace on ``device`` (call before capturing graphs)."""
    _P.workspace(torch.device(device), 0, 0)


# ----------------------------------------------------------------------------- workspace needs

def _need(M: int, N: int, K: int, ntw: int, splits: int) -> Tuple[int, int]:
    nc = 16 * ntw
    tiles = (N + nc - 1) // nc
    kchunk = ((K + splits - 1) // splits + 31) // 32 * 32
    S = (K + kchunk - 1) // kchunk
    # split-K slabs are laid out with the kernel's row-tile height (MT x 16 rows, MT in 1/2/4/8)
    mp = 16 * (1 if M <= 16 else 2 if M <= 32 else 4 if M <= 64 else 8)
    return (S * tiles * nc * mp if S > 1 else 0), tiles


def _need_dg(M: int, N: int, K: int, plan: Tuple[int, int, int]) -> Tuple[int, int]:
    """Floats and tickets of a decode GEMM ``plan``; (0, 0) where one workgroup has all of a tile's splits."""
    nt, vs, splits = plan
    kchunk = (-(-K // splits) + 31) // 32 * 32
    gy, tiles = -(-(-(-K // kchunk)) // vs), -(-N // (16 * nt))
    return (gy * vs * tiles * -(-M // 16) * 16 * (16 * nt + 1), tiles) if gy > 1 else (0, 0)


def _tg_splits(K: int, splits: int, ks: int = 1) -> int:
    q = 64 * ks
    kchunk = ((K + splits - 1) // splits + q - 1) // q * q
    return (K + kchunk - 1) // kchunk


def _need_tg(M: int, N: int, K: int, bm: int, bn: int, splits: int, ks: int = 1) -> Tuple[int, int]:
    tiles = ((M + bm - 1) // bm) * ((N + bn - 1) // bn)
    S = _tg_splits(K, splits, ks)
    return (S * tiles * bm * bn if S > 1 else 0), tiles


# ----------------------------------------------------------------------------- plans

def _heuristic(M: int, N: int, K: int, swiglu: bool = False) -> Tuple:
    """Plan of a shape nothing timed.  The splits of K depend on N and K alone and every split sums in the same order
    (skinny_gemm.hip), so up to 64 rows a row's bits depend neither on the batch nor on how the launch is cut: a design whose
    heads divide by small sums (mLSTM) turns a last bit into tenths of a logit.  What is left to choose is the columns of a
    workgroup (16 or 32) and ``_splits_together``.  K that is no whole 32s: the GEMV, which takes one, two and four rows."""
    if M > SKINNY_MAX_M:
        return ("blas",)
    if M > 64:
        tiles = (N + 15) // 16
        return ("skinny", 1, max(1, min(16, math.ceil(512 / tiles), K // 256)))
    if K % 32 and K % 8 == 0 and M in (1, 2, 4) and M * K * 2 <= 64 * 1024:
        return ("gemv", 1)
    splits = max(1, min(16, math.ceil(512 / ((N + 31) // 32)), K // 256))
    narrow = N * K <= _NARROW if M <= 32 else N <= 2048 and splits <= 4
    return ("skinny", 2 if swiglu else _apart(M, N, K, splits) or (1 if narrow else 2), splits)


# weights up to which 16 columns and four splits of K a workgroup (16 waves) beat 32 columns and two: past it the 16-wave workgroups,
# one a CU, come in several rounds.  us at 8 rows / 24 rows, 16 x 4, 32 x 2, and 32 x 1 as nothing else would choose:
# 1024 x 1024 4.2 / 5.1, 6.5 / 7.3, 6.1 / 6.7; 5632 x 1024 6.8 / 9.7, 8.6 / 11.9, 8.5 / 10.7; 1024 x 4096 11.4 / 12.7, 11.8 / 12.4,
# 12.4 / 13.2; 8192 x 2048 10.9 / 16.0, 10.8 / 12.7, 12.7 / 14.8.  Past 32 rows a workgroup re-reads more rows than weights: 16
# columns, a split each, where that is few workgroups (48 rows, 1024 x 1024: 7.1, 8.2, 8.5; 4096 x 1024 11.3, 8.9, 10.0).
_NARROW = 6 << 20


def _apart(M: int, N: int, K: int, splits: int) -> int:
    """Columns (in 16s) of a workgroup where more than four splits stay in workgroups of their own, else 0: few columns, whose joint
    workgroups are too few, and numbers of splits that leave a joint workgroup half empty.  us apart / together: 128 x 2048 8 rows 6.3 / 7.0,
    32 rows 7.2 / 8.8; 512 x 2048 8 rows 8.2 / 8.3, 32 rows 8.6 / 9.7, 64 rows 9.2 / 10.5; 256 x 8192 8 rows 11.0 (32 columns; 16 12.0) / 12.3; six splits:
    3000 x 1536 8 rows equal, 32 rows 11.0 / 12.6, 3000 x 4096 8 rows (32 columns) 11.5 / 13.1, 3000 x 8192 64 rows, 32 columns 32.9,
    16 38.2."""
    if splits <= 4:
        return 0
    if N <= 256 and splits > 8 and N > 128 and M <= 32:
        return 2
    if N <= 128 or (N <= 512 and M > 16):
        return 1
    if splits % 4 in (1, 2) and (M > 16 or N * K > _NARROW):
        return 1 if M > 16 and N * K <= 2 * _NARROW else 2
    return 0


def _splits_together(M: int, N: int, K: int, plan: Tuple) -> int:
    """Splits of K that share a workgroup of an untimed plan, meeting in LDS where they are all there (slabs and ticket cost 1.3 to 2.3
    us).  Three splits of 32 columns stay apart: the pairs would leave a quarter of the waves idle."""
    _, ntw, splits = plan
    if M > 64 or splits == 1 or _apart(M, N, K, splits):
        return 1
    if ntw == 1:
        return 4 if M <= 32 else 1
    return 1 if splits == 3 else 2


# Prefill-size buckets (M > MAX_M, PREFILL_TUNE): the fused ops' core is chosen per (bucket, N, K)
# between one tgemm launch with the epilogue fused and hipBLASLt + the standalone epilogue kernel;
# a prefill chunk uses the plan of the smallest bucket that holds it.  Rounds 4-5 measured it
# slower or neutral end to end (profiles/r4_prefill_gemm.md); with the grouped tile raster and the
# 8-loader 256 x 128 plans among the candidates (round 6) tgemm takes 8 of TinyLlama's 12 (bucket,
# shape) pairs (gate|up at 8K rows: 368 vs 448 us; 309 on four waves, csrc/kernels/wide_gemm.hip).  End to end it is within noise (+0.3 % over 7
# same-box arms of the driver command, prefill step time lower in 2 of 3; profiles/r6_prefill_core.md),
# and it is the default: the fused-epilogue kernel runs where it measured faster, hipBLASLt elsewhere.
PREFILL_MS = (2048, 4096, 8192)
PREFILL_TUNE = True
# decode buckets: the fused ops' core options are timed through the fused ops (_retime_fused)
FUSED_INSITU = True
# the split form (vendor / plain GEMM + standalone epilogue kernel) wins a fused op only when it is
# more than 3 % faster than the best one-launch core: on near-ties (QKV at the 512 bucket, 21-23 us
# either way in situ) the choice flipped run to run (profiles/r6_small_batch.md)
SPLIT_MARGIN = 1.03
# decode (v_new given): the standalone QKV epilogue hands V over row-major too, as the one-launch
# tgemm does, and the attention kernel writes the newest V^T (no 2-byte stores 32 B apart)
QKV_POST_VROWS = True
_PF_PLANS = ((256, 256, 2, 1, 1, 4), (256, 256, 2, 1, 1, 4, 1, 0, 0, 64, 16, 8),      # csrc/kernels/wide_gemm.hip
             (256, 128, 3, 1, 1, 8), (192, 128, 3, 1, 1, 8), (128, 128, 3, 1, 1, 8),
             # 32-deep k-steps: 5-13 % ahead of the 64-deep tiles at 2-4K rows (profiles/r5_decode_gemm_lab.md)
             (256, 256, 4, 1, 1, 8, 1, 0, 0, 32),
             # grouped tile raster (plan element 12: m-tiles per group), the 8-loader 256 x 128 tile: the
             # fastest tgemm forms at 2-8K rows in scripts/exp/raster_probe.py (profiles/r6_gemm_fill_path.md)
             (256, 256, 4, 1, 1, 8, 1, 0, 0, 32, 16, 8),
             (256, 128, 3, 1, 1, 8, 1, 8, 0, 64, 16, 0), (256, 128, 3, 1, 1, 8, 1, 8, 0, 64, 16, 2),
             (256, 128, 3, 1, 1, 8, 1, 8, 0, 64, 16, 8))


# Row counts between the decode buckets and the prefill buckets, whose plans are timed once too: a short prompt's products, and what
# prompt_parts leaves behind whole rounds of large tiles.
PF_SMALL_MS = (128, 256, 384, 512, 768, 1024)
PF_TAIL_MS = (1280, 1536, 1920, 2432, 3072, 3584, 3968)      # more of what is left (4096 rows of 2048 columns are a round of 256 x 128)
_PF_SMALL = ((64, 64, 3, 1, 1, 4), (64, 64, 3, 2, 1, 4), (64, 64, 4, 1, 1, 4, 1, 8), (64, 128, 3, 1, 1, 8), (128, 64, 4, 1, 1, 4, 1, 8),
             (128, 128, 3, 1, 1, 8), (160, 128, 3, 1, 1, 8, 1, 6), (192, 128, 3, 1, 1, 8), (256, 128, 3, 1, 1, 8, 1, 8))
_PART_US = 4.0            # a second launch of a product, and the clearing of row-sum slots it does not write
_PART_GAIN = 0.95         # another plan than the bucket's, or a second launch, where the rounds make it that much shorter: they are
#                           within 5 % of what is measured


def _small(m: int, N: int, K: int):
    """(fastest plan, its us) timed for the next of PF_SMALL_MS, or None."""
    b = next((b for b in PF_SMALL_MS if m <= b), None)
    return None if b is None else _P.pf_small.get((b, N, K))


def _left(m: int, N: int, K: int):
    """The same, of PF_TAIL_MS too."""
    b = next((b for b in PF_TAIL_MS if m <= b), None) if m > PF_SMALL_MS[-1] else None
    return _small(m, N, K) if b is None else _P.pf_tail.get((b, N, K))


def _rounds(tiles: int, cus: int) -> float:
    """Rounds that tiles take on the CUs: one that is part full is hardly shorter (TinyLlama's down, 256 x 128 and 192 x 128 tiles, 2100
    rows: 77 and 83 us with 144 and 176 of 256 CUs, 86 and 88 with all)."""
    full, rest = divmod(tiles, cus)
    return full + (0.8 + 0.2 * rest / cus if rest else 0.0)


def _round_us(N: int, K: int):
    """us a round of each timed prompt plan, from the largest size it was timed at."""
    out = {}
    for plan, m, t in sorted(_P.pf_times.get((N, K), ()), key=lambda e: e[1]):
        out[plan] = t / _rounds(-(-m // plan[0]) * -(-N // plan[1]), _P.cus)
    return out


def _parts_us(M: int, N: int, K: int) -> Tuple[float, Optional[Tuple]]:
    """(us, parts): ``prompt_parts`` worked out."""
    best, us, parts, cus = float("inf"), float("inf"), None, _P.cus
    rounds, usual = _round_us(N, K), tg_plan(M, N, K)
    tiles = lambda rows, plan: -(-rows // plan[0]) * -(-N // plan[1])
    if usual in rounds:
        us, parts = _rounds(tiles(M, usual), cus) * rounds[usual], ((M, usual),)
        best = _PART_GAIN * us
    for plan, u in rounds.items():
        t = _rounds(tiles(M, plan), cus) * u
        if t < best:
            best, us, parts = t, t, ((M, plan),)
        for k in range(1, -(-tiles(M, plan) // cus)):      # k rounds of it, and the rows they leave
            rows = k * cus // -(-N // plan[1]) * plan[0]
            tail = _left(M - rows, N, K) if 0 < rows < M else None
            if tail is not None:
                t = _rounds(tiles(rows, plan), cus) * u + tail[1] + _PART_US
                if t < best:
                    best, us, parts = t, t, ((rows, plan), (M - rows, tail[0]))
    return us, parts


def _keep(answers: dict, key, answer):
    if len(answers) > 4096:
        answers.clear()
    answers[key] = answer
    return answer


def prompt_parts(M: int, N: int, K: int) -> Optional[Tuple]:
    """How the one-launch form of a fused product of a prompt's M > MAX_M rows runs: ((rows, plan), ...) one behind the other, or None
    where nothing was timed.  A large tile costs by rounds over the CUs: 8928 rows of 2048 columns are 280 tiles of 256 x 256, two
    rounds of which the second holds 24, so the last 736 rows go to a launch of small tiles.  us, one launch / here, TinyLlama: Wo
    4500 rows 72 / 56, 8928 rows 140 / 94; gate|up 1500 rows 107 / 92, 3000 rows 196 / 157, 4500 rows 261 / 224.  What is left may be most of a
    round: past 1024 rows of it, the shortest of the other forms (the vendor's and its epilogue too) / here, 11679 rows: down 241 / 222, Wo
    109 / 102; QKV 8400 rows 100 / 87."""
    key = (M, N, K)
    if key in _P.pf_parts:
        return _P.pf_parts[key]
    parts = _parts_us(M, N, K)[1]
    return None if parts is None else _keep(_P.pf_parts, key, parts)


# Row counts beside the buckets at which the vendor's product and its epilogue are timed
PF_LIN_MS = (1280, 3072, 5120, 6144, 10240, 12288, 14336, 16384)
_VENDOR_GAIN = 0.97       # the other form than the bucket's, where it is that much shorter


def _vendor_at(M: int, N: int, K: int, bucket: bool) -> bool:
    """Whether a prompt's M rows run on the vendor's product and its epilogue: as their ``bucket``, unless the other form is the shorter one by
    what is timed around M.  Both go by rounds of tiles, of other sizes; between two timed sizes the vendor's takes as long as at the larger
    one, or longer.  us, vendor / one launch, TinyLlama: down 4500 rows 94 / 110, 8192 140 / 137, 8928 193 / 171, 10000 202 / 241, 11679 244 / 255,
    13000 246 / 241; output 4500 47 / 52, 8192 70 / 61, 10000 94 / 107, 11679 106 / 111; QKV 4096 58 / 72, 7000 104 / 100, 11679 138 / 136,
    14500 200 / 178.  Over 424 row counts of ten products this is 1.9 % above the shorter form, 3.2 % by the bucket alone."""
    key = (M, N, K)
    if key in _P.pf_vendor:
        return _P.pf_vendor[key]
    at, us = sorted(_P.pf_lin.get((N, K), ())), _parts_us(M, N, K)[0]
    if not at or us == float("inf"):
        return bucket
    lin = next((t for m, t in at if M <= m), at[-1][1] * M / at[-1][0])
    return _keep(_P.pf_vendor, key, us >= _VENDOR_GAIN * lin if bucket else lin < _VENDOR_GAIN * us)


# Plain products of prompts (layer lists): the row counts at which the vendor's is timed, and the tiles timed beside it at some of them
PP_MS = (*range(1280, 8193, 256), *range(8704, 12289, 512))
PP_OWN_MS = (2048, 4096, 8192, 12288)
_PP_PLANS = ((256, 256, 2, 1, 1, 4, 1, 0, 0, 64, 16, 8), (256, 128, 3, 1, 1, 8, 1, 8, 0, 64, 16, 8), (192, 128, 3, 1, 1, 8), (128, 128, 3, 1, 1, 8),
             (64, 128, 3, 1, 1, 8))
_PP_GAIN = 0.95           # estimates between timed sizes are within 5 % of what is measured


def prompt_plan(M: int, N: int, K: int, gelu: bool = False) -> Optional[Tuple]:
    """The tile on which M > MAX_M rows of x @ w.T [-> erf-GELU] run, or None: the vendor's product, or nothing was timed.  The vendor's time
    steps up and down with the rows: 13312 x 2048 271 us at 6144 rows, 366 to 373 from 6200 to 7424, 349 from 7500 to 8192 (here 256,
    291 to 316, 341 to 356), 6208 x 2048 111 at 5000, 190 at 7300, 155 at 7500 (105, 154, 152), 8192 x 2048 184 at 7308, 263 at 8193 (199, 242); so it is
    timed every few hundred rows, and taken to cost what it does at the next of them.  A tile's time goes by rounds over the CUs."""
    key = (M, N, K, int(gelu))
    if key in _P.pp_plans:
        return _P.pp_plans[key]
    vendor, own = _P.pp_times.get(key[1:], ((), ()))
    if not vendor or not own or M > 1.25 * vendor[-1][0]:
        return None
    us = next((t for m, t in vendor if M <= m), vendor[-1][1] * M / vendor[-1][0])
    m0, times = next((e for e in own if M <= e[0]), own[-1])
    best = None
    for plan, t in zip(_PP_PLANS, times):
        tiles = lambda m: -(-m // plan[0]) * -(-N // plan[1])
        t *= _rounds(tiles(M), _P.cus) / _rounds(tiles(m0), _P.cus)
        if 0 < t < _PP_GAIN * us and (best is None or t < best[0]):
            best = (t, plan)
    return _keep(_P.pp_plans, key, best and best[1])


def autotune_prompts(shapes: Iterable[Tuple[int, int, bool]], device, most: int = PP_MS[-1]) -> None:
    """Times the plain products of prompts, ``prompt_plan``'s choice: (N, K, with a GELU behind it) of each, up to the timed size that holds ``most``
    rows.  What was timed before stands.  Where there is no memory for a size, that and the longer ones are left to the vendor's product."""
    from . import seqmix
    dev = torch.device(device)
    if dev.type != "cuda" or most <= MAX_M or os.environ.get("DLLM_GEMM") == "blas":
        return
    cache = os.environ.get("DLLM_GEMM_PLANS")
    made = _timed_with(dev) if cache else ""
    if cache and os.path.exists(cache):
        _load_plans(cache, made)
    if _P.cus != _sk_grid(dev):
        _P.cus = _sk_grid(dev)
        _P.pf_parts.clear()
        _P.pf_vendor.clear()
        _P.pp_plans.clear()
    for N, K, gelu in shapes:
        key = (N, K, int(gelu))
        vendor, own = _P.pp_times.setdefault(key, ([], []))
        ms, own_ms = _pp_left(PP_MS, vendor, most), _pp_left(PP_OWN_MS, own, most)
        if not ms and not own_ms:
            continue
        try:
            copies = max(2, min(8, (256 << 20) // (N * K * 2)))
            ws = [torch.randn(N, K, dtype=torch.bfloat16, device=dev).mul_(0.02) for _ in range(copies)]
            for M in sorted({*ms, *own_ms}):
                x, y = torch.randn(M, K, dtype=torch.bfloat16, device=dev), torch.empty(M, N, dtype=torch.bfloat16, device=dev)

                def call(i):
                    torch.matmul(x, ws[i % copies].t(), out=y)
                    if gelu:
                        seqmix.gelu_erf(y)
                us = _time(call, iters=4) if M in ms else None
                if M in own_ms:
                    epi, ext = EPI_GELU if gelu else EPI_PLAIN, _native(x)
                    own.append((M, [_time(lambda i: _tgemm(ext, x, ws[i % copies], epi, p, y=y), iters=4) for p in _PP_PLANS]))
                if us is not None:
                    vendor.append((M, us))
                del x, y
        except torch.OutOfMemoryError:
            continue
        finally:
            for k in list(_P.pp_plans):      # (rows past what was timed have another answer now)
                if k[1:] == key:
                    _P.pp_plans.pop(k, None)
    if cache:
        _save_plans(cache, made)


def _pp_left(sizes: Iterable[int], have: list, most: int) -> List[int]:
    """The row counts that are left to time for prompts of up to ``most`` rows: up to the next one that holds them."""
    return [m for i, m in enumerate(sizes) if (i == 0 or sizes[i - 1] < most) and m > (have[-1][0] if have else 0)]


def prompt_gelu(x: torch.Tensor, w: torch.Tensor) -> Optional[torch.Tensor]:
    """``seqmix.gelu_erf(linear(x, w, prompt=True))`` in one launch where that is the faster form, else None."""
    plan = prompt_plan(x.shape[0], *w.shape, True) if _prompt_rows(x, w) else None
    if plan is None:
        return None
    y = torch.empty((x.shape[0], w.shape[0]), dtype=x.dtype, device=x.device)
    _tgemm(_native(x), x, w, EPI_GELU, plan, y=y)
    return y


def _prompt_rows(x: torch.Tensor, w: torch.Tensor) -> bool:
    """Rows and weights that the tiled GEMM reads, past the timed decode sizes."""
    return (x.is_cuda and x.shape[0] > MAX_M and x.dtype == w.dtype == torch.bfloat16 and x.dim() == 2 and x.stride(1) == 1 and x.stride(0) % 8 == 0 and
            x.stride(0) >= x.shape[1] and w.is_contiguous() and w.shape[1] % 64 == 0 and w.shape[0] % 8 == 0 and
            x.data_ptr() % 16 == 0 and w.data_ptr() % 16 == 0 and os.environ.get("DLLM_GEMM") != "blas")


def _row_parts(M: int, N: int, K: int, frag: bool = False) -> list:
    """[(first row, end, plan or "lin")]: a fused product's launches."""
    if use_vendor_core(M, N, K, True) if frag else use_vendor_core(M, N, K):
        return [(0, M, "lin")]
    parts = prompt_parts(M, N, K) if M > MAX_M and PREFILL_MS and not os.environ.get("DLLM_FUSED_CORE") else None
    out, lo = [], 0
    for rows, plan in parts or ((M, tg_plan(M, N, K)),):
        out.append((lo, lo + rows, plan))
        lo += rows
    return out


def prefill_bucket(M: int) -> int:
    for b in PREFILL_MS:
        if M <= b:
            return b
    return PREFILL_MS[-1] if PREFILL_MS else M


def next_batch_size(M: int) -> int:
    """The smallest decode batch size the engine times plans for (1, 2, 4, 8, 16, 32, 48, 64, then every 32 to 256, then every 64)
    that holds M rows.  A prompt of 57 tokens on TinyLlama: 1.37 ms of layer products with the plans
    of 64 rows against 1.58 with the untimed rule of ``tg_plan``."""
    for b in (1, 2, 4, 8, 16, 32, 48, 64):
        if M <= b:
            return b
    step = 32 if M <= 256 else 64
    return -(-M // step) * step


def tg_plan(M: int, N: int, K: int) -> Tuple[int, ...]:
    """(bm, bn, stages, splits, ks, waves[, k-groups]) of the fused GEMM for this shape: tuned, else a
    heuristic sized so the grid covers the 256 CUs (bigger tiles first, split-K only for short
    grids)."""
    p = _P.tg_plans.get((M, N, K))
    if p is None and M > MAX_M and PREFILL_MS:
        p = _P.tg_plans.get((prefill_bucket(M), N, K))
    if p is None and M <= MAX_M:      # rows between two timed batch sizes (a short prompt): what was timed for the next one
        p = _P.tg_plans.get((next_batch_size(M), N, K))
        if p is None and M > DG_MAX_M:
            p = (_small(M, N, K) or (None,))[0]
    if p is not None:
        return tuple(p) + (1, 4)[len(p) - 4:] if len(p) < 6 else tuple(p)
    mt64, nt64, nt128 = -(-M // 64), -(-N // 64), -(-N // 128)
    # 64 x 128 tiles of eight waves from 150 of them on, two workgroups a CU.  us 128 x 128 / here / 64 x 64 (GELU epilogue): 3800 rows
    # 1536 x 384 18 / 14 / 14, 384 x 1536 21 / 15 / 17, 8000 rows 1536 x 384 29 / 24 / 33, 1200 rows 3072 x 2048 27 / 25 / 32, 16000 rows 4096 x
    # 1024 260 / 232 / 292, 500 rows 1536 x 384 9 / 7 / 7; at 500 rows of 1152 x 1536 (72 tiles) 21 / 14 / 12.  More columns than rows are few
    # tiles of many rows' worth of weights: 300 rows of 4096 x 4096 (160) 43 / 30 / 28, 600 of 2304 x 768 (180) 15 / 10.8 / 10.3, 600 of
    # 3072 x 768 (240) 15 / 11.2 / 11.3.  A long K down to fewer columns (residual epilogue) reads less with 128 x 128, where its tiles are
    # whole rounds: 1024 x 4096, 4000 rows (256 tiles) 45 / 49, 8000 89 / 97, 2000 (128) 41 / 30; 4096 x 4096, 2000 rows 88 / 92; 768 x 3072,
    # 16000 rows (750) 104 / 108, 8000 (378) 64 / 57
    tiles = -(-M // 128) * nt128
    if K >= 2048 and N <= K and tiles >= 0.9 * _P.cus * -(-tiles // _P.cus):
        return (128, 128, 3, 1, 1, 8)
    if mt64 * nt128 >= (150 if M >= N else 185):
        return (64, 128, 3, 1, 1, 8)
    tiles = mt64 * nt64
    splits = 1
    while tiles * splits * 2 <= 512 and K // (splits * 2) >= 256 and splits < 8:
        splits *= 2
    if _need_tg(M, N, K, 64, 64, splits)[0] > WS_FLOATS:
        splits = 1
    return (64, 64, 3, splits, 1, 4)


def tg_slots(M: int, N: int, K: int) -> int:
    """Row-sum-of-squares slots a RESADD GEMM of this shape writes (one per n-tile)."""
    return -(-N // tg_plan(M, N, K)[1])


def _run_plan(plan, x, w, swiglu, out, wp=None, together=1):
    if plan[0] == "blas":
        if swiglu:
            x = ref_silu_mul(x)
        return torch.matmul(x, w.t(), out=out) if out is not None else F.linear(x, w)
    ext = _native(x)
    if plan[0] == "tg":
        if swiglu:
            x = ref_silu_mul(x)
        y = out if out is not None else torch.empty((x.shape[0], w.shape[0]), dtype=x.dtype, device=x.device)
        _tgemm(ext, x, wp if wp is not None else w, EPI_PLAIN, plan[1:], y=y)
        return y
    if plan[0] == "gemv":
        y = out if out is not None else torch.empty((x.shape[0], w.shape[0]), dtype=x.dtype, device=x.device)
        ext.gemv(x, w, y, plan[1], swiglu)
        return y
    kind, ntw, splits = plan
    M, N, K = x.shape[0], w.shape[0], w.shape[1]
    y = out if out is not None else torch.empty((M, N), dtype=x.dtype, device=x.device)
    floats, tiles = _need(M, N, K, ntw, splits)
    part, cnt = _P.workspace(x.device, floats, tiles)
    ext.skinny_gemm(x, w, y, ntw, splits, swiglu, part, cnt, together)
    return y


def stream_k_table(M: int, N: int, K: int, bm: int, bn: int, ks: int, grid: int):
    """Stream-K work split of an (M, N, K) GEMM over ``grid`` workgroups (csrc/kernels/tgemm.hip,
    GemmArgs.sk_table): the tiles x k-steps iteration space is cut into ``grid`` equal contiguous
    ranges; workgroup w walks its range as segments (tile, first k-step, end k-step, slab index |
    contributors << 16).  A tile covered by c workgroups gets slab indices 0..c-1 in k order, so its
    last arriver sums the partials in the same order every time.  Returns (int32 [grid, segmax, 4]
    array padded with tile -1, cmax = the largest contributor count)."""
    import numpy as np
    mt, nt = -(-M // bm), -(-N // bn)
    tiles, nkt = mt * nt, K // (64 * ks)
    total = tiles * nkt
    segs = [[] for _ in range(grid)]
    contrib: Dict[int, list] = {}
    for w in range(grid):
        it, hi = w * total // grid, (w + 1) * total // grid
        while it < hi:
            t, kb = divmod(it, nkt)
            ke = min(nkt, kb + hi - it)
            segs[w].append([t, kb, ke, 0])
            contrib.setdefault(t, []).append((w, len(segs[w]) - 1))
            it += ke - kb
    cmax = max(len(v) for v in contrib.values())
    for t, lst in contrib.items():
        for idx, (w, j) in enumerate(lst):
            segs[w][j][3] = idx | (len(lst) << 16)
    segmax = max(1, max(len(s_) for s_ in segs))
    tab = np.full((grid, segmax, 4), -1, dtype=np.int32)
    for w, sl in enumerate(segs):
        if sl:
            tab[w, :len(sl)] = np.asarray(sl, dtype=np.int32)
    return tab, cmax


def _sk_grid(dev) -> int:
    return torch.cuda.get_device_properties(dev).multi_processor_count


def _sk_tensor(dev, M, N, K, bm, bn, ks):
    """The device copy of a stream-K table, created once per shape outside graph capture (the
    engine's capture warm-up runs every step eagerly first) and kept for the process lifetime."""
    key = (str(dev), M, N, K, bm, bn, ks)
    hit = _P.sk_tables.get(key)
    if hit is None:
        if torch.cuda.is_current_stream_capturing():
            raise RuntimeError("stream-K table first needed during graph capture (run the step eagerly first)")
        tab, cmax = stream_k_table(M, N, K, bm, bn, ks, _sk_grid(dev))
        hit = (torch.from_numpy(tab).to(dev), cmax)
        _P.sk_tables[key] = hit
    return hit


def _tgemm(ext, x, w, epi, plan, y=None, ssq_in=None, ssq_n=0, norm_scale=0.0, eps=0.0, ssq_out=None,
           pos=None, cos_sin=None, slots=None, q_out=None, kc=None, vc=None, nq=0, nkv=0, d=0, bias=None,
           v_rows=None):
    """plan = (bm, bn, stages, splits[, ks, waves[, k-groups[, loader waves[, stream-K[, k depth[, mfma[, raster]]]]]]])"""
    bm, bn, st, sp = plan[:4]
    ks, nw = (plan[4], plan[5]) if len(plan) >= 6 else (1, 4)
    wk = plan[6] if len(plan) >= 7 else 1
    nl = plan[7] if len(plan) >= 8 else 0
    sk = len(plan) >= 9 and plan[8] == 1
    bk = plan[9] if len(plan) >= 10 else 64
    mf = plan[10] if len(plan) >= 11 else 16
    raster = plan[11] if len(plan) >= 12 else 0
    if sk and epi != EPI_PLAIN:
        raise ValueError("tgemm: stream-K plans are built for the PLAIN epilogue only")
    M = x.shape[0]
    N, K = _nk(w)
    if K % (64 * ks):
        ks, wk = 1, 1
    part = cnt = tab = None
    cmax = 0
    if sk:
        tab, cmax = _sk_tensor(x.device, M, N, K, bm, bn, ks)
        tiles = -(-M // bm) * -(-N // bn)
        part, cnt = _P.workspace(x.device, tiles * cmax * bm * bn, tiles)
        sp = 1
    elif _tg_splits(K, sp, ks) > 1:
        floats, tiles = _need_tg(M, N, K, bm, bn, sp, ks)
        part, cnt = _P.workspace(x.device, floats, tiles)
    ext.tgemm(x, w, y, epi, bm, bn, st, sp, ks, nw, part, cnt, ssq_in, int(ssq_n), float(norm_scale), float(eps), ssq_out,
              pos, cos_sin, slots, q_out, kc, vc, int(nq), int(nkv), int(d), bias, int(wk), int(nl), tab, int(cmax),
              v_rows, int(bk), int(mf), int(raster))


def ref_silu_mul(gu):
    from . import silu_mul
    return silu_mul(gu)


def _key(x, w, swiglu):
    return (x.shape[0], w.shape[0], w.shape[1], bool(swiglu))


def dgemm(x: torch.Tensor, wf: torch.Tensor, n: int, epi: int, plan: Tuple[int, int, int], y=None, res=None, ssq_out=None,
          scale: float = 0.0, eps: float = 0.0, pos=None, cos_sin=None, slots=None, q_out=None, kc=None, vc=None, v_rows=None,
          nq: int = 0, nkv: int = 0, d: int = 0, bias=None, mode: int = 0, limit: float = 0.0, alpha: float = 1.0) -> int:
    """One launch of the decode GEMM on ``wf`` = frag_weight of an [n, K] weight; ``plan`` = (16-column tiles a workgroup, splits a
    workgroup, splits of K)."""
    nt, vs, splits = plan
    floats, tiles = _need_dg(x.shape[0], n, x.shape[1], plan)
    part, cnt = _P.workspace(x.device, floats, tiles) if floats else (None, None)
    return int(_native(x).dgemm(x, wf, n, int(epi), nt, vs, splits, y, part, cnt, res, ssq_out, float(scale), float(eps), pos, cos_sin,
                                slots, q_out, kc, vc, v_rows, int(nq), int(nkv), int(d), bias, int(mode), float(limit), float(alpha)))


def dg_takes(x: torch.Tensor) -> bool:
    """The decode GEMM reads these rows: up to 64, 16-byte aligned."""
    return 0 < x.shape[0] <= DG_MAX_M and x.dtype == torch.bfloat16 and x.stride(1) == 1 and x.stride(0) % 8 == 0 and \
        (x.shape[0] == 1 or x.stride(0) >= x.shape[1]) and x.data_ptr() % 16 == 0


FG_MAX_M, FG_MAX_K = 16, 8192      # f32_gemm.hip: past them the vendor GEMM is as fast


def _fg_wins(M: int, N: int, K: int) -> bool:
    """Past eight rows the vendor GEMM is ahead on wide and on long products, us vendor / here: 16 rows 8192 x 2048 15.9 / 19.7, 32000 x 1536
    44 / 52, 128 x 2048 6.8 / 7.5, 32000 x 512 17.2 / 17.7, 1024 x 4096 10.8 / 14.7; but 4096 x 2048 12.6 / 11.5, 8192 x 1024 12.7 / 10.7, 12 rows 32000 x 1024 34.7 / 32.7.
    Up to eight it is nowhere."""
    if M <= 8:
        return True
    return (N <= 16384 or M <= 12) if K <= 1024 else 512 <= N <= 4096 and K <= 2048


def fg_takes(x: torch.Tensor, N: Optional[int] = None) -> bool:
    """The f32 decode product reads these rows: up to 16, 16-byte aligned; ``N``: and is the faster one for N columns."""
    return 0 < x.shape[0] <= FG_MAX_M and x.dtype == torch.float32 and x.dim() == 2 and x.stride(1) == 1 and x.stride(0) % 4 == 0 and \
        (x.shape[0] == 1 or x.stride(0) >= x.shape[1]) and x.data_ptr() % 16 == 0 and os.environ.get("DLLM_GEMM") != "blas" and \
        (N is None or _fg_wins(x.shape[0], N, x.shape[1]))


def f32_linear(x: torch.Tensor, wf: torch.Tensor, N: int, gelu: bool = False) -> torch.Tensor:
    """``x @ w.T`` [-> erf-GELU] of up to 16 f32 rows on the weight's fragment-major copy (csrc/kernels/f32_gemm.hip)."""
    y = torch.empty((x.shape[0], N), dtype=torch.float32, device=x.device)
    _native(x).f32_gemm(x, wf, y, DG_GELU if gelu else EPI_PLAIN)
    return y


def _linear_plan(x: torch.Tensor, w: torch.Tensor, frag: bool, keep_order: bool, ends: bool = False):
    """(plan on the row-major weight, splits a workgroup, decode GEMM's plan or None) of ``linear``; ``ends``: the decode GEMM would end in
    the activation, a launch (3.4 us) that the plan it is timed against has yet to make."""
    M, (N, K) = x.shape[0], w.shape
    plan, together = _P.plans.get(_key(x, w, False)), 1
    dg = _P.dg_plans.get((M, N, K)) if frag and not keep_order else None
    timed = plan is not None
    if not timed:
        plan = _heuristic(M, N, K) if M <= MAX_M else ("blas",)
    if plan[0] == "skinny":
        same = ("skinny", min(plan[1], 2), plan[2])
        as_one = _splits_together(M, N, K, same)
        if not timed:
            together = as_one
        if frag and dg is None and (not timed or keep_order or ends):
            dg = (same[1], as_one, same[2])
            floats, tiles = _need_dg(M, N, K, dg)
            if M > DG_MAX_M or floats > WS_FLOATS or tiles > WS_COUNTERS:      # (a slab is a column wider than the skinny plan's)
                dg = None
    return plan, together, dg


def linear_act(x: torch.Tensor, w: torch.Tensor, wf: torch.Tensor, act: str, bias: Optional[torch.Tensor] = None, limit: float = 0.0,
               alpha: float = 1.0, keep_order: bool = False) -> Optional[torch.Tensor]:
    """``seqmix.gelu_erf(linear(x, w))`` (act "gelu") or ``seqmix.glu_act(linear(x, w), bias, act, limit, alpha)`` in the launch of the
    decode GEMM, where it takes the product; else None.  ``wf``: frag_weight(w), paired = "glu" for the gated ones."""
    if not dg_takes(x) or os.environ.get("DLLM_GEMM") == "blas":
        return None
    dg = _linear_plan(x, w, True, keep_order, ends=True)[2]
    if dg is None:
        return None
    N = w.shape[0]
    y = torch.empty((x.shape[0], N if act == "gelu" else N // 2), dtype=x.dtype, device=x.device)
    if act == "gelu":
        dgemm(x, wf, N, DG_GELU, dg, y=y)
    else:
        from .seqmix import GLU_MODES
        dgemm(x, wf, N, DG_GLU, dg, y=y, bias=bias, mode=GLU_MODES[act], limit=limit, alpha=alpha)
    return y


TAIL_MAX_M, TAIL_MAX_K = 16, 1024      # tail_gemm.hip: rows and width of what a workgroup norms


class Tail:
    """A sublayer's tail that the product behind it takes along (csrc/kernels/tail_gemm.hip): ``x2 = x + rmsnorm(y + bias) * w_post``
    (f32, another buffer than x), and the product's input ``rmsnorm(x2) * w_next``, which exists nowhere else.  Goes where that input
    would (``shape``, ``device``, ``dtype`` are its own)."""

    def __init__(self, y, w_post, eps, x, x2, w_next, bias=None):
        self.y, self.w_post, self.eps, self.x, self.x2, self.w_next, self.bias = y, w_post, eps, x, x2, w_next, bias
        self.shape, self.device, self.dtype, self.is_cuda = y.shape, y.device, y.dtype, y.is_cuda

    def linear(self, w: torch.Tensor, wf: torch.Tensor, act: Optional[str] = None, act_bias: Optional[torch.Tensor] = None,
               limit: float = 0.0, alpha: float = 1.0) -> torch.Tensor:
        """``linear`` of the input, or with ``act`` ``linear_act``'s gated form; once, and on the engine's stream before x2 is read."""
        from .seqmix import GLU_MODES
        N = w.shape[0]
        out = torch.empty((self.shape[0], N if act is None else N // 2), dtype=self.dtype, device=self.device)
        _native(self.y).tail_gemm(self.y, self.x, self.x2, self.w_post, self.w_next, self.bias, float(self.eps), wf, N, out,
                                  1 if N <= 16 * _sk_grid(self.device) else 2, act is not None, act_bias,
                                  0 if act is None else GLU_MODES[act], float(limit), float(alpha))
        return out


def tail_takes(y: torch.Tensor, w: torch.Tensor, *vectors: Optional[torch.Tensor]) -> bool:
    """Does a ``Tail`` of y go into the product with w [N, K] (which has a fragment-major copy)?  Up to 16 rows of at most 1024, and
    columns for one round of workgroups: each norms every row.  ``vectors``: the f32 vectors it reads."""
    M, (N, K) = y.shape[0], w.shape
    return (y.is_cuda and y.dtype == torch.bfloat16 and 0 < M <= TAIL_MAX_M and y.shape[1] == K <= TAIL_MAX_K and K % 32 == 0 and
            y.stride(1) == 1 and y.stride(0) % 4 == 0 and (M == 1 or y.stride(0) >= K) and y.data_ptr() % 8 == 0 and
            N <= 32 * _sk_grid(y.device) and os.environ.get("DLLM_GEMM") != "blas" and
            all(v is None or (v.dtype == torch.float32 and v.is_contiguous() and v.data_ptr() % 16 == 0) for v in vectors))


def tail_wins(M: int, K: int) -> bool:
    """Is one launch the faster form?  From the 13th row on a SIMD norms four, which widths up to 512 do not bear: us, two launches / one, 3136 columns, 8,
    12, 13 and 16 rows of 256 5.4 / 4.8, 5.5 / 5.5, 5.4 / 5.9, 5.5 / 6.1; of 512 6.0 / 4.8, 6.1 / 5.5, 6.1 / 6.0, 6.1 / 6.3; of 576 6.2 / 4.8, 6.3 / 5.7,
    6.2 / 6.0, 6.5 / 6.4; of 768 and 16 6.7 / 6.4."""
    return M <= 12 or K > 512


def linear(x: torch.Tensor, w: torch.Tensor, out: Optional[torch.Tensor] = None,
           wp: Optional[torch.Tensor] = None, wf: Optional[torch.Tensor] = None, keep_order: bool = False, prompt: bool = False) -> torch.Tensor:
    """``x @ w.T`` on the shape's tuned plan; ``prompt``: many rows may take the tile timed for them (``prompt_plan``); ``wp``: the panel copy a tgemm plan streams, ``wf``: the fragment-major copy of the
    decode GEMM, which takes the untimed products of up to 64 rows with the splits and the order of sums they have without it, and
    timed ones where it was faster, or with ``keep_order`` where the plan is a skinny one, whose sums it keeps."""
    if not x.is_cuda or os.environ.get("DLLM_GEMM") == "blas":
        return F.linear(x, w) if out is None else torch.matmul(x, w.t(), out=out)
    tile = prompt_plan(x.shape[0], *w.shape) if prompt and _prompt_rows(x, w) else None
    if tile is not None:
        return _run_plan(("tg",) + tile, x, w, False, out)
    plan, together, dg = _linear_plan(x, w, wf is not None, keep_order)
    if dg is not None and dg_takes(x):
        y = out if out is not None else torch.empty((x.shape[0], w.shape[0]), dtype=x.dtype, device=x.device)
        dgemm(x, wf, w.shape[0], EPI_PLAIN, dg, y=y)
        return y
    return _run_plan(plan, x, w, False, out, wp, together)


def norm_linear(h: torch.Tensor, residual: torch.Tensor, spare: torch.Tensor, norm_w: torch.Tensor, eps: float,
                w: torch.Tensor) -> Tuple[torch.Tensor, torch.Tensor]:
    """``linear(rmsnorm(h + residual) * norm_w, w)`` and the updated residual stream (unfused
    layer path: tensor parallel, CPU).  (A one-launch GEMV form, gemv.hip NORM, measured SLOWER at
    batch 1, profiles/r1_small_batch_decode.md; ``spare`` is kept for that interface.)"""
    from . import rms_norm
    x = rms_norm(h, norm_w, eps, residual=residual)
    return linear(x, w), residual


def linear_swiglu(gu: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """``silu(gate) * up @ w.T`` with gu = [gate | up] of width 2K."""
    if not gu.is_cuda:
        return F.linear(ref.silu_mul(gu), w)
    if gu.shape[0] > MAX_M or os.environ.get("DLLM_GEMM") == "blas":
        from . import silu_mul
        return linear(silu_mul(gu), w)
    plan = _P.plans.get(_key(gu, w, True)) or _heuristic(gu.shape[0], w.shape[0], w.shape[1], True)
    return _run_plan(plan, gu, w, True, None)


# ----------------------------------------------------------------------------- fused decoder ops
#
# Two implementations of each fused op: the tgemm epilogue (one launch), or the shape's best plain
# GEMM (GEMV / skinny / hipBLASLt, whatever the autotuner picked for linear()) followed by the same
# epilogue as a standalone kernel (qkv_post / res_add_ssq / swiglu_post).
# The autotuner records, per decode bucket and shape, which is faster (the standalone epilogue
# is charged its measured time, _post_us; POST_US only where it cannot be measured); shapes it never saw (prefill chunks above MAX_M) use the vendor core,
# which wins at large M (profiles/r2_tgemm_tune.md).
POST_US = 3.0


def _core_of(M: int, N: int, K: int, frag: bool) -> Optional[str]:
    """The timed core of a fused op whose weight has (``frag``) or has no fragment-major copy; a decode GEMM is ``fused_dg``'s to take,
    rows it does not read get what was chosen without it."""
    c = _P.frag_core.get((M, N, K)) if frag else None
    return _P.fused_core.get((M, N, K)) if c is None or c.startswith("dg") else c


def use_vendor_core(M: int, N: int, K: int, frag: bool = False) -> bool:
    """True: run the fused op as ``linear()`` (the shape's best plain plan — GEMV / skinny /
    hipBLASLt / plain tgemm) followed by the standalone epilogue kernel; False: one tgemm launch
    with the epilogue fused.  (A ``gemvR`` choice is taken before this by ``fused_gemv_r``.)"""
    env = os.environ.get("DLLM_FUSED_CORE")
    if env in ("tg", "blas", "lin"):
        return env != "tg"
    c = _core_of(M, N, K, frag)
    if c is None and M > MAX_M and PREFILL_MS:
        c = _P.fused_core.get((prefill_bucket(M), N, K))
        if c is not None:
            return _vendor_at(M, N, K, c != "tg")
    if c is not None:
        return c != "tg"
    return M > MAX_M


def fused_gemv_r(x: torch.Tensor, N: int, frag: bool = False) -> int:
    """R (output rows per wave) of the fused-epilogue GEMV (csrc/kernels/gemv.hip EPI) if the
    autotuner picked it for this fused op's shape (``fused_core`` = ``gemvR``; forced by
    ``DLLM_FUSED_CORE=gemvR``), else 0.  Batch <= 8 only: it replaces GEMV/skinny + a standalone
    epilogue launch (qkv_post / res_add_ssq / swiglu_post) with one launch."""
    M, K = x.shape[0], x.shape[1]
    if M not in _GEMV_MS or K % 8 or M * K * 2 > 64 * 1024 or x.stride(1) != 1 or x.stride(0) % 8 or N % 32:
        return 0
    env = os.environ.get("DLLM_FUSED_CORE")
    c = env if env else _core_of(M, N, K, frag)
    if isinstance(c, str) and c.startswith("gemv") and c[4:] in ("1", "2", "4"):
        return int(c[4:])
    return 0


def fused_ske(x: torch.Tensor, N: int, K: int, frag: bool = False) -> int:
    """Split count of the small-batch fused-epilogue MFMA GEMM (skinny_epi, 32-column tiles) if the
    autotuner picked it for this fused op's shape (``fused_core`` = ``skE<splits>``; forced by
    ``DLLM_FUSED_CORE=skE<splits>``), else 0."""
    M = x.shape[0]
    if not (0 < M <= SKE_MAX_M) or K % 64 or N % 32 or x.stride(1) != 1 or x.stride(0) % 8:
        return 0
    env = os.environ.get("DLLM_FUSED_CORE")
    c = env if env and env.startswith("skE") else _core_of(M, N, K, frag)
    if isinstance(c, str) and c.startswith("skE") and c[3:].isdigit():
        return int(c[3:])
    return 0


def _ske_ws(x: torch.Tensor, N: int, K: int, splits: int):
    tiles = -(-N // 32)
    kchunk = ((-(-K // splits)) + 31) // 32 * 32
    S = -(-K // kchunk)
    return _P.workspace(x.device, (S * tiles * 32 * 16) if S > 1 else 0, tiles)


def skinny_epi(x: torch.Tensor, w: torch.Tensor, epi: int, splits: int, y=None, res=None, ssq_out=None, ssq_in=None,
               ssq_n: int = 0, scale: float = 0.0, eps: float = 0.0, pos=None, cos_sin=None, slots=None, q_out=None,
               kc=None, vc=None, nq: int = 0, nkv: int = 0, d: int = 0) -> int:
    """One launch of the small-batch fused-epilogue GEMM (``w`` row-major or the panel copy)."""
    N, K = _nk(w)
    part, cnt = _ske_ws(x, N, K, splits)
    return int(_native(x).skinny_epi(x, w, y, 2, int(splits), int(epi), part, cnt, res, ssq_out, ssq_in, int(ssq_n),
                                     float(scale), float(eps), pos, cos_sin, slots, q_out, kc, vc, int(nq), int(nkv),
                                     int(d)))


def fused_dg(x: torch.Tensor, N: int, K: int, wf: Optional[torch.Tensor]) -> Optional[Tuple[int, int, int]]:
    """Plan of the decode GEMM (csrc/kernels/decode_gemm.hip) if the autotuner picked it for this fused op's shape (``frag_core`` =
    ``dg<nt>.<vs>.<splits>``) and the caller keeps its weight copy, else None."""
    if wf is None:
        return None
    M = x.shape[0]      # rows between two timed batch sizes (a short prompt): what was timed for the next one
    c = os.environ.get("DLLM_FUSED_CORE") or _P.frag_core.get((M, N, K)) or _P.frag_core.get((next_batch_size(M), N, K))
    if not c or not c.startswith("dg") or not dg_takes(x):
        return None
    return tuple(int(v) for v in c[2:].split("."))


def _core(x: torch.Tensor, w: torch.Tensor, wp: Optional[torch.Tensor] = None) -> torch.Tensor:
    """Plain product for the split (core + epilogue) form of a fused op: the tuned plan of this
    shape (M <= MAX_M), hipBLASLt above."""
    return linear(x, w, wp=wp) if x.shape[0] <= MAX_M else F.linear(x, w)

def qkv_rope_cache(r: torch.Tensor, w: torch.Tensor, ssq: torch.Tensor, ssq_n: int, eps: float,
                   positions: torch.Tensor, cos_sin: torch.Tensor, slots: torch.Tensor, k_cache: torch.Tensor,
                   v_cache: torch.Tensor, nq: int, nkv: int, d: int, wp: Optional[torch.Tensor] = None,
                   v_new: Optional[torch.Tensor] = None, wf: Optional[torch.Tensor] = None):
    """q [T, nq, d] of ``rope(rmsnorm(r) . Wqkv^T)``, K/V written to the paged caches, one launch.

    ``w`` is the folded/permuted weight of models.llama.fuse_qkv_weight; ``ssq[:ssq_n]`` holds
    the partial row sums of r^2 written by the producer of ``r``.

    ``v_new`` ([T, nkv * d], decode steps only): where the one-launch GEMM runs, V is written there
    row-major instead of into the V^T cache, and the decode attention kernel moves each sequence's
    newest V into the cache itself (``paged_attention(v_new=...)``: the GEMM's V-column workgroups
    were its stragglers, profiles/r5_qkv_epilogue.md).  Returns ``(q, v_new or None)`` then — None
    where another implementation ran and the cache already holds V."""
    T, H = r.shape
    q = torch.empty((T, nq, d), dtype=r.dtype, device=r.device)
    if T == 0:
        return q if v_new is None else (q, None)
    out = (lambda used: q if v_new is None else (q, v_new if used else None))
    dg = fused_dg(r, w.shape[0], H, wf)
    if dg:
        dgemm(r, wf, w.shape[0], EPI_QKV, dg, scale=1.0 / H, eps=eps, pos=positions, cos_sin=cos_sin, slots=slots, q_out=q, kc=k_cache,
              vc=v_cache, v_rows=v_new, nq=nq, nkv=nkv, d=d)
        return out(True)
    R = fused_gemv_r(r, w.shape[0], wf is not None)
    if R:
        _native(r).gemv_qkv(r, w, ssq, int(ssq_n), 1.0 / H, float(eps), positions, cos_sin, slots, q, k_cache,
                            v_cache, nq, nkv, d, R)
        return out(False)
    sp = fused_ske(r, w.shape[0], H, wf is not None)
    if sp:
        skinny_epi(r, wp if wp is not None else w, EPI_QKV, sp, ssq_in=ssq, ssq_n=ssq_n, scale=1.0 / H, eps=eps,
                   pos=positions, cos_sin=cos_sin, slots=slots, q_out=q, kc=k_cache, vc=v_cache, nq=nq, nkv=nkv, d=d)
        return out(False)
    for lo, hi, plan in _row_parts(T, w.shape[0], H, wf is not None):
        rows, sq = (r, ssq) if hi - lo == T else (r[lo:hi], ssq[:, lo:hi])
        if plan == "lin":
            vr = v_new if QKV_POST_VROWS else None
            _native(r).qkv_post(_core(rows, w, wp), sq, int(ssq_n), 1.0 / H, float(eps), positions[lo:hi], cos_sin, slots[lo:hi], q[lo:hi],
                                k_cache, v_cache, nq, nkv, d, vr)      # (all rows)
            used = vr is not None
        else:
            _tgemm(_native(r), rows, wp if wp is not None else w, EPI_QKV, plan, ssq_in=sq, ssq_n=ssq_n, norm_scale=1.0 / H,
                   eps=eps, pos=positions[lo:hi], cos_sin=cos_sin, slots=slots[lo:hi], q_out=q[lo:hi], kc=k_cache, vc=v_cache, nq=nq,
                   nkv=nkv, d=d, v_rows=v_new if v_new is None else v_new[lo:hi])
            used = True
    return out(used)


def matmul_resadd(x: torch.Tensor, w: torch.Tensor, residual: torch.Tensor, ssq_out: torch.Tensor,
                  wp: Optional[torch.Tensor] = None, wf: Optional[torch.Tensor] = None) -> int:
    """``residual += x . w^T`` (bf16 rounding as ``rms_norm``'s residual add) and the partial row
    sums of the new residual's squares into ``ssq_out[:slots]``; returns ``slots``."""
    M, N, K = x.shape[0], w.shape[0], w.shape[1]
    dg = fused_dg(x, N, K, wf) if M else None
    if dg:
        return dgemm(x, wf, N, EPI_RESADD, dg, res=residual, ssq_out=ssq_out)
    R = fused_gemv_r(x, N, wf is not None) if M else 0
    if R:
        return int(_native(x).gemv_resadd(x, w, residual, ssq_out, R))
    sp = fused_ske(x, N, K, wf is not None) if M else 0
    if sp:
        return skinny_epi(x, wp if wp is not None else w, EPI_RESADD, sp, res=residual, ssq_out=ssq_out)
    if not M:
        return -(-N // tg_plan(M, N, K)[1])
    parts = _row_parts(M, N, K, wf is not None)
    if parts[0][2] == "lin":
        return int(_native(x).res_add_ssq(_core(x, w, wp), residual, ssq_out))
    n = max(-(-N // p[1]) for _, _, p in parts)
    for lo, hi, plan in parts:
        mine, whole = -(-N // plan[1]), hi - lo == M
        so = ssq_out if whole else ssq_out[:, lo:hi]
        _tgemm(_native(x), x if whole else x[lo:hi], wp if wp is not None else w, EPI_RESADD, plan, y=residual if whole else residual[lo:hi],
               ssq_out=so)
        if mine < n:
            so[mine:n].zero_()
    return n


def swiglu_matmul(r: torch.Tensor, w: torch.Tensor, ssq: torch.Tensor, ssq_n: int, eps: float,
                  wp: Optional[torch.Tensor] = None, wf: Optional[torch.Tensor] = None) -> torch.Tensor:
    """``silu(g) * u`` with ``[g | u] = rmsnorm(r) . Wgu^T`` (interleaved rows, models.llama
    .fuse_gate_up_weight) -> [T, I]."""
    T, H = r.shape
    act = torch.empty((T, w.shape[0] // 2), dtype=r.dtype, device=r.device)
    dg = fused_dg(r, w.shape[0], H, wf) if T else None
    if dg:
        dgemm(r, wf, w.shape[0], EPI_SWIGLU, dg, y=act, scale=1.0 / H, eps=eps)
        return act
    R = fused_gemv_r(r, w.shape[0], wf is not None) if T else 0
    if R:
        _native(r).gemv_swiglu(r, w, ssq, int(ssq_n), 1.0 / H, float(eps), act, R)
        return act
    sp = fused_ske(r, w.shape[0], H, wf is not None) if T else 0
    if sp:
        skinny_epi(r, wp if wp is not None else w, EPI_SWIGLU, sp, y=act, ssq_in=ssq, ssq_n=ssq_n, scale=1.0 / H,
                   eps=eps)
        return act
    if not T:
        return act
    for lo, hi, plan in _row_parts(T, w.shape[0], H, wf is not None):
        rows, sq = (r, ssq) if hi - lo == T else (r[lo:hi], ssq[:, lo:hi])
        if plan == "lin":
            _native(r).swiglu_post(_core(rows, w, wp), sq, int(ssq_n), 1.0 / H, float(eps), act[lo:hi])
        else:
            _tgemm(_native(r), rows, wp if wp is not None else w, EPI_SWIGLU, plan, y=act[lo:hi], ssq_in=sq, ssq_n=ssq_n, norm_scale=1.0 / H,
                   eps=eps)
    return act


def res_add_ssq(h: Optional[torch.Tensor], r: torch.Tensor, ssq: torch.Tensor) -> int:
    """``r += h`` in place (h may be None) and the row sums of ``r^2``: ``ssq`` [M] gets the full
    sum, ``ssq`` [slots, >= M] partial sums over column slices.  Returns the slots written."""
    return int(_native(r).res_add_ssq(h, r, ssq))


# ----------------------------------------------------------------------------- encoder (bias) ops

def _enc_ok(x: torch.Tensor, w: torch.Tensor) -> bool:
    return x.is_cuda and w.shape[1] % 64 == 0 and w.shape[0] % 8 == 0 and x.stride(1) == 1 and x.stride(0) % 8 == 0


def linear_bias(x: torch.Tensor, w: torch.Tensor, bias: torch.Tensor, gelu: bool = False) -> torch.Tensor:
    """``x . w^T + bias`` (optionally followed by erf-GELU) in one tgemm launch (bias / GELU
    epilogue): the router encoder's QKV and FFN-up projections."""
    if not _enc_ok(x, w):
        y = F.linear(x, w, bias)
        return ref.gelu(y) if gelu else y
    M, N, K = x.shape[0], w.shape[0], w.shape[1]
    y = torch.empty((M, N), dtype=x.dtype, device=x.device)
    epi = EPI_GELU if gelu else EPI_PLAIN
    if M and not _native(x).enc_gemm(x, w, bias, y, epi):      # few rows: straight to registers, else the tiled GEMM
        _tgemm(_native(x), x, w, epi, tg_plan(M, N, K), y=y, bias=bias)
    return y


def linear_bias_residual(x: torch.Tensor, w: torch.Tensor, bias: torch.Tensor, residual: torch.Tensor) -> torch.Tensor:
    """``residual += x . w^T + bias`` in place (tgemm residual epilogue with bias; bf16 rounding of
    the projection before the add, as F.linear followed by an add); returns ``residual``."""
    if not _enc_ok(x, w):
        residual.copy_((F.linear(x, w, bias).float() + residual.float()).to(residual.dtype))
        return residual
    M, N, K = x.shape[0], w.shape[0], w.shape[1]
    if M and not _native(x).enc_gemm(x, w, bias, residual, EPI_RESADD):
        _tgemm(_native(x), x, w, EPI_RESADD, tg_plan(M, N, K), y=residual, bias=bias)
    return residual


def encoder_layers(x: torch.Tensor, lens: torch.Tensor, starts: torch.Tensor, S: int, nh: int, d: int, eps: float,
                   layers) -> torch.Tensor:
    """The sentence encoder's layers (dicts with wqkv, bqkv, wo, bo, ln1, w1, b1, w2, b2, ln2) over packed rows x [T, nh d], which
    are overwritten: QKV, attention, output + residual, LayerNorm, up + GELU, down + residual, LayerNorm.  On the GPU one call
    launches them all."""
    from . import encoder_attention, layer_norm
    plan = _encoder_plan(x, layers)
    if plan:
        return _native(x).encoder_layers(x, lens, starts, int(S), int(nh), int(d), float(eps), *plan)
    for L in layers:
        a = encoder_attention(linear_bias(x, L["wqkv"], L["bqkv"]), lens, lens.numel(), S, nh, d, starts=starts)
        x = layer_norm(linear_bias_residual(a, L["wo"], L["bo"], x), *L["ln1"], eps)
        f = linear_bias(x, L["w1"], L["b1"], gelu=True)
        x = layer_norm(linear_bias_residual(f, L["w2"], L["b2"], x), *L["ln2"], eps)
    return x


def encoder_texts(ids: torch.Tensor, at: torch.Tensor, emb, lens: torch.Tensor, starts: torch.Tensor, S: int, nh: int, d: int, eps: float,
                  layers) -> torch.Tensor:
    """Unit vectors [B, nh d] (f32) of packed texts: embeddings (``emb``: word, pos, type0, norm w, b), ``encoder_layers``, mean over each text's
    rows.  On the GPU one call, whose first and last launches hold the embeddings (up to 16 rows) and the mean."""
    from . import embed_ln, mean_pool_l2
    T, word = ids.numel(), emb[0]
    # past 16 rows a launch of its own, under way while this call is prepared (inside it 96 texts took 10 us more)
    few = T <= 16 and word.is_cuda
    x = torch.empty((T, word.shape[1]), dtype=word.dtype, device=word.device) if few else embed_ln(ids, *emb, S, eps, at)
    plan = _encoder_plan(x, layers)
    if not plan:
        x = embed_ln(ids, *emb, S, eps, at) if few else x
        return mean_pool_l2(encoder_layers(x, lens, starts, S, nh, d, eps, layers), lens, starts)
    out = torch.empty((lens.numel(), word.shape[1]), dtype=torch.float32, device=word.device)
    _native(x).encoder_layers(x, lens, starts, int(S), int(nh), int(d), float(eps), *plan, [ids, at, *emb] if few else [], out)
    return out


def _encoder_plan(x: torch.Tensor, layers):
    """Weights, plans and scratch of the native encoder on rows like x (None: not its shapes)."""
    T, names = x.shape[0], ("wqkv", "wo", "w1", "w2")
    if not (T and layers and x.is_contiguous() and all(_enc_ok(x, L[n]) for L in layers for n in names)):
        return None
    shapes = [tuple(layers[0][n].shape) for n in names]
    plans = [tg_plan(T, n, k) for n, k in shapes]
    if any(tuple(L[n].shape) != s for L in layers for n, s in zip(names, shapes)) or any(p[8:9] == (1,) for p in plans):
        return None
    full, floats, tiles = [], 0, 0
    for p, (n, k) in zip(plans, shapes):
        p = p + (1, 4, 1, 0, 0, 64, 16, 0)[len(p) - 4:]
        if k % (64 * p[4]):
            p = p[:4] + (1, p[5], 1) + p[7:]
        if _tg_splits(k, p[3], p[4]) > 1:
            fl, ti = _need_tg(T, n, k, p[0], p[1], p[3], p[4])
            floats, tiles = max(floats, fl), max(tiles, ti)
        full.append(list(p[:8] + p[9:]))
    part, cnt = _P.workspace(x.device, floats, tiles) if tiles else (None, None)
    weights = [t for L in layers for t in (L["wqkv"], L["bqkv"], L["wo"], L["bo"], *L["ln1"], L["w1"], L["b1"], L["w2"], L["b2"], *L["ln2"])]
    return weights, full, part, cnt


def max_slots(N: int, M: int = 0) -> int:
    """Rows a partial-row-sum buffer needs for a residual producer of N columns: one per 64-column
    tgemm tile, at batch <= 8 one per fused-GEMV workgroup (N / 4 at R = 1), at batch <= 64 one
    per 16-column tile of the decode GEMM."""
    if 0 < M <= max(_GEMV_MS):
        return -(-N // 4)
    return -(-N // 16) if 0 < M <= DG_MAX_M else -(-N // 64)


# ----------------------------------------------------------------------------- autotuning

def _time(fn, iters=24) -> float:
    """GPU time per call of fn(i) in us, measured as a hipGraph replay of ``iters`` calls (the
    decode step is a graph replay too, so host launch cost is excluded exactly as in serving).
    Callers rotate operands over i so weights come from HBM, not the 256 MiB Infinity Cache."""
    fn(0)  # eager warm-up: initialises libraries outside capture
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    st = torch.cuda.Stream()
    st.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(st):
        with torch.cuda.graph(g, stream=st):
            for i in range(iters):
                fn(i)
    torch.cuda.current_stream().wait_stream(st)
    g.replay()
    torch.cuda.synchronize()
    s, e = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    s.record()
    g.replay()
    e.record()
    torch.cuda.synchronize()
    return s.elapsed_time(e) * 1000.0 / iters


def _post_us(M: int, N: int, dev) -> float:
    """Measured cost of the standalone epilogue a vendor-core fused op adds: one pass reading two
    [M, N] bf16 operands and writing one (res_add_ssq; qkv_post / swiglu_post move the same or
    fewer bytes).  Charged to hipBLASLt when choosing the fused op's core."""
    if N % 8:
        return POST_US
    y = torch.zeros(M, N, dtype=torch.bfloat16, device=dev)
    r = torch.zeros(M, N, dtype=torch.bfloat16, device=dev)
    ssq = torch.empty(max_slots(N), M, dtype=torch.float32, device=dev)
    ext = _native(y)
    return _time(lambda i: ext.res_add_ssq(y, r, ssq))


def _plan_key(k) -> str:
    if len(k) == 3:
        return "t,%d,%d,%d" % k
    return "%d,%d,%d,%d" % (k[0], k[1], k[2], int(k[3]))


# A plan file's key beside its plans: what they were timed with.  Times hold for the kernels that were timed, a choice for the candidates it
# was made among: a file from before a kernel or a candidate plan would keep both out for good.
_TIMED_WITH = "timed with"


def _timed_with(dev) -> str:
    """The candidates (this file), the kernels as built, the vendor's library and the device."""
    import hashlib
    h = hashlib.sha1()
    for path in (__file__, getattr(_load_ext(), "__file__", "")):
        if path and os.path.exists(path):
            with open(path, "rb") as f:
                h.update(f.read())
    p = torch.cuda.get_device_properties(dev)
    # (not by its name, which is empty under a profiler)
    return "%s %s %d %s" % (torch.__version__, p.gcnArchName, p.multi_processor_count, h.hexdigest())


def _load_plans(path: str, timed_with: Optional[str] = None) -> None:
    """``timed_with``: nothing of a file that was timed with anything else (None: any file)."""
    with open(path) as f:
        d = json.load(f)
        if d.pop(_TIMED_WITH, None) != timed_with and timed_with is not None:
            return
        for k, v in d.items():
            kind, *at = k.split(",")
            if kind == "t":
                _P.tg_plans[tuple(map(int, at))] = tuple(v)
            elif kind == "s":
                _P.pf_small[tuple(map(int, at))] = (tuple(v[0]), v[1])
            elif kind == "e":
                _P.pf_tail[tuple(map(int, at))] = (tuple(v[0]), v[1])
            elif kind == "l":
                _P.pf_lin[tuple(map(int, at))] = [tuple(e) for e in v]
            elif kind == "m":
                _P.pp_times[tuple(map(int, at))] = ([tuple(e) for e in v[0]], [(m, list(t)) for m, t in v[1]])
            elif kind == "p":
                _P.pf_times[tuple(map(int, at))] = [(tuple(q), m, t) for q, m, t in v]
            elif kind == "d":
                _P.dg_plans[tuple(map(int, at))] = v and tuple(v)
            elif kind == "r":
                _P.frag_core[tuple(map(int, at))] = v
            elif kind == "c":
                if not v.startswith("dg"):      # (files that kept one choice for weights with and without copies: timed again)
                    _P.fused_core[tuple(map(int, at))] = v
            else:
                _P.plans[(int(kind), int(at[0]), int(at[1]), at[2] == "1")] = tuple(v)


def _save_plans(path: str, timed_with: str = "") -> None:
    d = {_plan_key(k): list(v) for k, v in _P.plans.items()}
    d.update({_plan_key(k): list(v) for k, v in _P.tg_plans.items()})
    d.update({"c,%d,%d,%d" % k: v for k, v in _P.fused_core.items()})
    d.update({"r,%d,%d,%d" % k: v for k, v in _P.frag_core.items()})
    d.update({"d,%d,%d,%d" % k: v and list(v) for k, v in _P.dg_plans.items()})
    d.update({"s,%d,%d,%d" % k: list(v) for k, v in _P.pf_small.items()})
    d.update({"e,%d,%d,%d" % k: list(v) for k, v in _P.pf_tail.items()})
    d.update({"p,%d,%d" % k: v for k, v in _P.pf_times.items()})
    d.update({"l,%d,%d" % k: v for k, v in _P.pf_lin.items()})
    d.update({"m,%d,%d,%d" % k: v for k, v in _P.pp_times.items()})
    d[_TIMED_WITH] = timed_with
    if os.path.dirname(path):
        os.makedirs(os.path.dirname(path), exist_ok=True)
    with open(path, "w") as f:
        json.dump(d, f)


def autotune(shapes: Iterable[Tuple[int, int, bool]], ms: Iterable[int], device, verbose: bool = False,
             fused: Iterable[Tuple[int, int]] = (), prefill: bool = False, qkv_dims=None, qkv_cache=None,
             frag: Iterable[Tuple[int, int]] = ()) -> None:
    """Measure every candidate plan for each (M, N, K, swiglu) and keep the fastest.

    ``fused``: the (N, K) shapes of one decoder layer's fused ops (QKV, Wo, gate|up, down); a
    residual producer keeps the fused GEMV only where its consumer runs it too
    (``_couple_gemv_choices``).  Their fused-op cores are timed through the fused ops themselves
    (``_retime_fused``); ``qkv_dims`` = (nq, nkv, d) of the QKV op (None: QKV keeps the stand-in
    timings); ``qkv_cache`` = one layer's (K, V^T) caches of the engine, which the QKV timing writes
    into at scattered free blocks (the TLB reach of a whole serving pool, not of a small buffer); ``frag`` =
    the (N, K) shapes whose weights have fragment-major copies (the decode GEMM is then a candidate)."""
    dev = torch.device(device)
    if dev.type != "cuda" or os.environ.get("DLLM_GEMM") == "blas":
        return
    reserve(dev)
    if _P.cus != _sk_grid(dev):
        _P.cus = _sk_grid(dev)
        _P.pf_parts.clear()
        _P.pf_vendor.clear()
        _P.pp_plans.clear()
    cache = os.environ.get("DLLM_GEMM_PLANS")  # JSON plan cache: re-use a previous run's choices
    made = _timed_with(dev) if cache else ""
    if cache and os.path.exists(cache):
        _load_plans(cache, made)
    shapes = list(shapes)
    fused = list(fused)
    # the fused ops' tgemm plans stream the panel weight copies: time them in that layout
    roles = {}
    if len(fused) in (2, 4):   # (QKV, Wo[, gate|up, down]) of a layer
        roles = dict(zip((tuple(f) for f in fused), ("qkv", "resadd", "swiglu", "resadd")))
    _autotune(shapes, list(ms), dev, verbose, {tuple(f) for f in fused} if W_PANEL else set(), roles, qkv_dims,
              qkv_cache, {tuple(f) for f in frag})
    _couple_gemv_choices(fused, list(ms), verbose)
    if PREFILL_TUNE or prefill:
        _autotune_prefill(fused, dev, verbose, roles, qkv_dims)
    if cache:
        _save_plans(cache, made)


def _autotune_prefill(fused, dev, verbose: bool, roles=None, qkv_dims=None) -> None:
    """Fused-op core at the prefill buckets: one tgemm launch with the epilogue fused against hipBLASLt + the standalone epilogue kernel,
    both timed through the fused op (by their plain products TinyLlama's QKV of 4096 rows went to one launch of 72 us from
    58; where a shape has no fused op: PLAIN, and the vendor's plus ``_post_us``), the vendor's at PF_LIN_MS as well (``_vendor_at``);
    the tgemm plans stream the K-panel weight copy the model keeps (W_PANEL).  Plans of the sizes below the buckets are timed too."""
    roles = roles or {}
    for (N, K) in {tuple(f) for f in fused}:
        todo = [M for M in PREFILL_MS if (M, N, K) not in _P.fused_core]
        if not todo or K % 64:
            continue
        copies = max(2, min(8, (256 << 20) // (N * K * 2)))
        ws = [(torch.randn(N, K, device=dev) * 0.02).to(torch.bfloat16) for _ in range(copies)]
        wps = [panel_weight(w) for w in ws] if W_PANEL else ws
        lins = {}
        for M in sorted({*todo, *PF_LIN_MS}) if (N, K) in roles else ():
            try:
                whole = _fused_call(roles[(N, K)], torch.randn(M, K, device=dev).to(torch.bfloat16), ws, wps, qkv_dims, dev)
                _P.fused_core[(M, N, K)] = "lin"
                lins[M] = _time(whole, iters=8)
            except Exception:  # noqa: BLE001 - no such fused op, or no memory for so many rows
                continue
            finally:
                _P.fused_core.pop((M, N, K), None)
        _P.pf_lin[(N, K)] = sorted({**dict(_P.pf_lin.get((N, K), ())), **lins}.items())
        for M in todo:
            x = torch.randn(M, K, device=dev).to(torch.bfloat16)
            y = torch.empty(M, N, dtype=torch.bfloat16, device=dev)
            ext = _native(x)
            lin = lins.get(M) or _time(lambda i: torch.matmul(x, ws[i % copies].t(), out=y), iters=8) + _post_us(M, N, dev)
            best, best_t, best_whole = None, float("inf"), float("inf")
            times = _P.pf_times.setdefault((N, K), [])
            whole = _fused_call(roles.get((N, K)), x, ws, wps, qkv_dims, dev)
            for p in _PF_PLANS:
                try:
                    t = t_whole = _time(lambda i: _tgemm(ext, x, wps[i % copies], EPI_PLAIN, p, y=y), iters=8)
                    if whole is not None:      # with its epilogue: what choosing among the plans goes by
                        _P.pf_parts[(M, N, K)], _P.fused_core[(M, N, K)] = ((M, p),), "tg"
                        t_whole = _time(whole, iters=8)
                except Exception:  # noqa: BLE001 - plan refused for this shape
                    continue
                finally:
                    _P.pf_parts.pop((M, N, K), None)
                    _P.fused_core.pop((M, N, K), None)      # (not timed yet: ``todo``)
                if t < best_t:
                    best, best_t = p, t
                best_whole = min(best_whole, t_whole)
                times.append((p, M, t_whole))
            if best is not None:
                _P.tg_plans[(M, N, K)] = best
            _P.fused_core[(M, N, K)] = "tg" if best_whole < lin else "lin"
            if verbose:
                print(f"gemm prefill M={M} N={N} K={K}: blas+post {lin:.1f}us, tgemm {best} {best_whole:.1f}us "
                      f"-> {_P.fused_core[(M, N, K)]}", flush=True)
            del x, y
        res: dict = {}
        for M in PF_SMALL_MS + PF_TAIL_MS:
            x, y = torch.randn(M, K, device=dev).to(torch.bfloat16), torch.empty(M, N, dtype=torch.bfloat16, device=dev)
            far = {p for p, t in res.items() if M in PF_TAIL_MS and t > 1.6 * min(res.values())}      # at the size before: not timed again
            ext, res = _native(x), {}
            for p in _PF_SMALL:
                if p in far or p[0] > max(64, M) or (p[3] > 1 and _need_tg(M, N, K, p[0], p[1], p[3])[0] > WS_FLOATS) or _tg_splits(K, p[3]) != p[3]:
                    continue
                try:
                    res[p] = _time(lambda i: _tgemm(ext, x, wps[i % copies], EPI_PLAIN, p, y=y), iters=8)
                except Exception:  # noqa: BLE001 - plan refused for this shape
                    continue
            best = min(res, key=res.get, default=None)
            if best is not None:
                (_P.pf_small if M in PF_SMALL_MS else _P.pf_tail)[(M, N, K)] = (best, res[best])
            if verbose and best is not None:
                print(f"gemm rows M={M} N={N} K={K}: {best} {res[best]:.1f}us", flush=True)
        _P.pf_parts.clear()
        _P.pf_vendor.clear()
        del ws, wps


def _couple_gemv_choices(fused, ms, verbose: bool) -> None:
    """A fused-GEMV residual producer leaves one row-sum slot per workgroup (hundreds), which a
    GEMV consumer sums in one round trip but a tgemm prologue or standalone epilogue walks
    serially.  ``fused`` = (QKV, Wo, gate|up, down) shapes of a dense layer: Wo feeds gate|up and
    down feeds the next layer's QKV, so a producer keeps the GEMV only if its consumer runs it too
    (MoE layers pass (QKV, Wo): their producers feed standalone norms, no constraint)."""
    fused = list(fused)
    pairs = [(fused[1], fused[2]), (fused[3], fused[0])] if len(fused) == 4 else []
    # the decode GEMM's narrowest tiles leave a slot per 16 columns; as a consumer it takes the row sums from its own operands
    for cores, many, fits, out in ((_P.fused_core, ("gemv",), ("gemv", "skE"), ("gemv", "dg")),
                                   (_P.frag_core, ("gemv", "dg1."), ("gemv", "skE", "dg"), ("gemv", "dg1."))):
        for M in ms:
            for prod, cons in pairs:
                kp, kc = (M,) + tuple(prod), (M,) + tuple(cons)
                cp, cc = cores.get(kp), cores.get(kc, _P.fused_core.get(kc))
                if cp is None or not cp.startswith(many) or (cc is not None and cc.startswith(fits)):
                    continue
                opts = {c: t for c, t in _P.fused_opts.get(kp, {}).items() if not c.startswith(out)}
                cores[kp] = min(opts, key=opts.get) if opts else "lin"
                if verbose:
                    print(f"gemm M={M} N={kp[1]} K={kp[2]}: {cp} dropped (its consumer N={kc[1]} K={kc[2]} "
                          f"runs {cc}, which would walk the per-workgroup row sums) -> core {cores[kp]}",
                          flush=True)


def _tg_cands(M: int, N: int, K: int):
    if K % 64:
        return []
    out = []
    for bm, bn, nw in _TG_TILES:
        if (bm == 128 and M <= 64) or (bm >= 192 and M <= 128):
            continue
        tiles = -(-M // bm) * -(-N // bn)
        for ks in (1, 2):
            if K % (64 * ks):
                continue
            for sp in _TG_SPLITS:
                if sp > 1 and (K // sp < 256 * ks or tiles * sp > 2048):
                    continue
                if _tg_splits(K, sp, ks) != sp:
                    continue
                if _need_tg(M, N, K, bm, bn, sp, ks)[0] > WS_FLOATS:
                    continue
                for st in ((2, 3, 4, 6) if bm <= 128 and ks == 1 else (2, 3)):
                    if st * ks * (bm + bn) * 128 > 150 * 1024:
                        continue   # the ring would not fit the LDS
                    out.append((bm, bn, st, sp, ks, nw))
                    if ks == 2 and nw == 4 and st <= 3 and bm <= 128 and bn <= 128:
                        out.append((bm, bn, st, sp, ks, nw, 2))   # two k-groups of 4 waves
    if N % 8 == 0:
        for bm, bn, nw, st, nl, m_min in _TG_NL:
            if M < m_min or (bm == 16 and M > 16):
                continue
            tiles = -(-M // bm) * -(-N // bn)
            for sp in (1, 2, 3, 4):
                if sp > 1 and (K // sp < 256 or tiles * sp > 2048 or _tg_splits(K, sp) != sp):
                    continue
                if _need_tg(M, N, K, bm, bn, sp)[0] > WS_FLOATS:
                    continue
                out.append((bm, bn, st, sp, 1, nw, 1, nl))
    # 32 x 32 x 16 MFMA forms of the flagship's tiles, with the splits their 16 x 16 forms take
    if N % 8 == 0:
        for p in _TG_M32:
            bm, bn, st, _, ks, nw, wk, nl = p[:8]
            if (bm >= 128 and M <= 64) or (bm == 256 and M <= 128) or K % (64 * ks):
                continue
            tiles = -(-M // bm) * -(-N // bn)
            for sp in (1, 2, 3, 4):
                if sp > 1 and (K // sp < 256 * ks or tiles * sp > 2048 or _tg_splits(K, sp, ks) != sp):
                    continue
                if _need_tg(M, N, K, bm, bn, sp, ks)[0] > WS_FLOATS:
                    continue
                out.append((bm, bn, st, sp) + tuple(p[4:]))
    # Stream-K forms (one workgroup per CU walking equal shares of tiles x k-steps, _SK_PLANS) are not
    # offered: measured, they never beat the one-unit plans on the TinyLlama shapes at M = 320-448,
    # because the shared-operand L2 -> LDS traffic, not the idle CUs, sets the time
    # (profiles/r3_decode_gemm_panel.md section 5).  They stay built for the PLAIN epilogue (tests).
    return [c for c in out if tg_built(c)]


def _dg_cands(M: int, N: int, K: int):
    """(nt, vs, splits) of the decode GEMM worth timing: a wave walks at least 64 k, the grid is no more than eight workgroups a CU and
    not under a quarter of the CUs."""
    out = []
    if M > DG_MAX_M or K % 32:
        return out
    for nt in (1, 2, 3):
        for vs in (1, 2):
            for gy in (1, 2, 4) if nt < 3 else (1,):      # three tiles a workgroup: where the weight is wide
                s, tiles = vs * gy, -(-N // (16 * nt))
                kchunk = (-(-K // s) + 31) // 32 * 32
                if -(-K // kchunk) != s or K // (4 * s) < 64 or not 64 <= tiles * gy <= 2048 or (gy > 1 and tiles * gy > 1024):
                    continue
                if _need_dg(M, N, K, (nt, vs, s))[0] > WS_FLOATS:
                    continue
                out.append((nt, vs, s))
    return out


def _fused_call(role, x, ws, wps, qkv_dims, dev, qkv_cache=None, wfs=None):
    """fn(i): the fused op of a layer's weight (``role`` qkv, resadd or swiglu) on rows x and the i-th copy of its weights, or None."""
    if role is None:
        return None
    M, N, K = x.shape[0], ws[0].shape[0], ws[0].shape[1]
    copies = len(ws)
    wsrc = lambda i: (ws[i % copies], wps[i % copies] if wps is not None else None)
    wf = lambda i: wfs[i % copies] if wfs is not None else None
    prompt = M > MAX_M
    slots_in = -(-K // (128 if prompt else 32))   # the producer's partial row sums (as many as a skinny_epi producer leaves)
    ssq = torch.rand(slots_in, M, device=dev) + 1.0
    if role == "resadd":
        res = torch.zeros(M, N, dtype=torch.bfloat16, device=dev)
        so = torch.empty(max_slots(N, M), M, dtype=torch.float32, device=dev)
        fn = lambda i: matmul_resadd(x, wsrc(i)[0], res, so, wp=wsrc(i)[1], wf=wf(i))
    elif role == "swiglu":
        fn = lambda i: swiglu_matmul(x, wsrc(i)[0], ssq, slots_in, 1e-5, wp=wsrc(i)[1], wf=wf(i))
    elif role == "qkv" and qkv_dims is not None:
        nq, nkv, d = qkv_dims
        if (nq + 2 * nkv) * d != N:
            return None
        # the step writes each row's K / V into its own block of a large pool: scattered slots in the
        # engine's own cache (else a 64 MiB pool; contiguous slots in a tiny cache timed the split
        # form's K / V^T writes 3.5 us per call faster than they run in the flagship's step)
        if (qkv_cache is not None and tuple(qkv_cache[0].shape[1:]) == (nkv, 16, d)
                and qkv_cache[0].shape[0] >= M + 1):
            kc, vc = qkv_cache
            nblk = kc.shape[0]
        else:
            nblk = max(-(-M // 16) + 1, (64 << 20) // (nkv * 16 * d * 2))
            kc = torch.zeros(nblk, nkv, 16, d, dtype=torch.bfloat16, device=dev)
            vc = torch.zeros(nblk, nkv, d, 16, dtype=torch.bfloat16, device=dev)
        pos = torch.randint(100, 4000, (M,), dtype=torch.int32, device=dev)
        if prompt:      # one sequence's rows, one behind the other
            sl = torch.arange(M, dtype=torch.int32, device=dev)
        else:
            sl = (torch.randperm(nblk, device=dev)[:M] * 16 + torch.randint(0, 16, (M,), device=dev)).to(torch.int32)
        cs = torch.rand(4096, d, device=dev)
        # (d = 64 decode hands V over row-major, as models.llama does: the one-launch cores then skip
        # the strided V^T cache writes)
        vn = torch.empty(M, nkv * d, dtype=torch.bfloat16, device=dev) if d == 64 and not prompt else None
        fn = lambda i: qkv_rope_cache(x, wsrc(i)[0], ssq, slots_in, 1e-5, pos, cs, sl, kc, vc, nq, nkv, d,
                                      wp=wsrc(i)[1], v_new=vn, wf=wf(i))
    else:
        return None
    return fn


def _retime_fused(tkey, role, opts, x, ws, wps, qkv_dims, dev, qkv_cache=None, wfs=None):
    """Time every fused-core option of a decoder-layer shape through the fused op itself: its real
    epilogue and its row-scale prologue over the producer's partial row sums.  The stand-in timings
    (PLAIN tgemm, RESADD GEMV / skinny_epi) missed those: gate|up at batch 4 chose a tgemm timed at
    13.6 us that ran 17.3 us inside the step graph (profiles/r6_small_batch.md)."""
    M, N, K = tkey
    if wfs is not None:
        opts = dict(opts, **{"dg%d.%d.%d" % p: 0.0 for p in _dg_cands(M, N, K)})
    fn = _fused_call(role, x, ws, wps, qkv_dims, dev, qkv_cache, wfs)
    if fn is None:
        return None
    cores = _P.fused_core if wfs is None else _P.frag_core
    saved = cores.get(tkey)
    out = {}
    try:
        for _ in range(2):   # two interleaved passes, the faster of each option's two times
            for opt in opts:
                cores[tkey] = opt
                try:
                    t = _time(fn)
                except Exception:  # noqa: BLE001 - option not runnable for this shape
                    t = float("inf")
                out[opt] = min(out.get(opt, float("inf")), t)
    finally:
        if saved is None:
            cores.pop(tkey, None)
        else:
            cores[tkey] = saved
    return out


def _best_core(opts: Dict[str, float]) -> str:
    core = min(opts, key=opts.get)
    one = {c: t for c, t in opts.items() if c != "lin"}
    if core == "lin" and one and min(one.values()) <= SPLIT_MARGIN * opts["lin"]:
        core = min(one, key=one.get)
    return core


def _time_dg(tkey, us: float, x, wfs) -> None:
    """Time the decode GEMM's candidates on the copies ``wfs`` of a shape's weights; ``us``: the plan to beat."""
    M, N, K = tkey
    y = torch.empty(M, N, dtype=torch.bfloat16, device=x.device)
    t = {p: _time(lambda i: dgemm(x, wfs[i % len(wfs)], N, EPI_PLAIN, p, y=y)) for p in _dg_cands(M, N, K)}
    best = min(t, key=t.get, default=None)
    _P.dg_plans[tkey] = best if best is not None and t[best] < us else None
    if _P.dg_plans[tkey]:
        _P.timings.setdefault((M, N, K, False), {})["dg"] = round(t[best], 2)


def _time_frag_core(tkey, role, x, ws, wps, qkv_dims, dev, qkv_cache, wfs) -> None:
    """The decode GEMM against the core that was chosen where there were no copies."""
    opts = _retime_fused(tkey, role, {_P.fused_core[tkey]: 0.0}, x, ws, wps, qkv_dims, dev, qkv_cache, wfs)
    if opts:
        _P.fused_opts.setdefault(tkey, {}).update(opts)
        _P.frag_core[tkey] = _best_core(opts)


def _autotune(shapes, ms, dev, verbose: bool, panel_shapes=frozenset(), roles=None, qkv_dims=None,
              qkv_cache=None, frag_shapes=frozenset()) -> None:
    use_tg = True
    for (N, K, sw) in shapes:
        copies = max(2, min(64, math.ceil((768 << 20) / (N * K * 2))))
        ws = [(torch.randn(N, K, device=dev) * 0.02).to(torch.bfloat16) for _ in range(copies)]
        wps = [panel_weight(w) for w in ws] if (N, K) in panel_shapes and K % 64 == 0 and not sw else None
        wfs = [frag_weight(w) for w in ws] if (N, K) in frag_shapes and K % 32 == 0 and not sw else None
        for M in ms:
            if M > MAX_M:
                continue
            key = (M, N, K, sw)
            tkey = (M, N, K)
            need_plain = key not in _P.plans
            need_tg = use_tg and not sw and (tkey not in _P.tg_plans or tkey not in _P.fused_core) and K % 64 == 0
            role = (roles or {}).get((N, K)) if FUSED_INSITU and M <= MAX_M and os.environ.get("DLLM_FUSED_CORE") is None else None
            # with copies there is more to choose from; what was chosen without them stands
            need_dg = wfs is not None and M <= DG_MAX_M and tkey not in _P.dg_plans
            need_frag = wfs is not None and M <= DG_MAX_M and role is not None and K % 64 == 0 and tkey not in _P.frag_core
            if not (need_plain or need_tg or need_dg or need_frag):
                continue
            x = torch.randn(M, 2 * K if sw else K, device=dev).to(torch.bfloat16)
            plain = lambda c: _time(lambda i: _run_plan(c, x, ws[i % copies], sw, None, wps[i % copies] if wps is not None else None))  # noqa: E731
            if not (need_plain or need_tg):
                if need_dg:
                    _time_dg(tkey, plain(_P.plans[key]), x, wfs)
                if need_frag:
                    _time_frag_core(tkey, role, x, ws, wps, qkv_dims, dev, qkv_cache, wfs)
                continue
            cands = [("blas",)]
            if M in _GEMV_MS and K % 8 == 0 and M * K * 2 <= 64 * 1024:
                cands.extend(("gemv", r) for r in _GEMV_RS)
            for ntw in (_NTWS if M <= SKINNY_MAX_M else ()):
                if M > 64 and ntw == 4:
                    continue
                for s in _SPLITS:
                    if s > 1 and K // s < 128:
                        continue
                    floats, tiles = _need(M, N, K, ntw, s)
                    if floats > WS_FLOATS or tiles > WS_COUNTERS:
                        continue
                    cands.append(("skinny", ntw, s))
            if use_tg and not sw:
                cands.extend(("tg",) + c for c in _tg_cands(M, N, K))
            res = {c: plain(c) for c in cands}
            best = min(res, key=res.get)
            if need_plain:
                _P.plans[key] = best
                _P.timings[key] = {str(c): round(t, 2) for c, t in res.items()}
            if need_dg:
                _time_dg(tkey, res[_P.plans[key]] if _P.plans[key] in res else res[best], x, wfs)
            tgc = [c for c in res if c[0] == "tg"]
            post = None
            if need_tg and tgc:
                best_tg = min(tgc, key=res.get)
                _P.tg_plans[tkey] = best_tg[1:]
                post = _post_us(M, N, dev)
                # the split form runs the shape's best plain plan (GEMV at M <= 8, skinny, ...)
                best_plain = min(res[c] for c in res if c[0] != "tg")
                opts = {"tg": res[best_tg], "lin": best_plain + post}
                # fused-epilogue GEMV (one launch): timed in its RESADD form (the paired QKV /
                # SwiGLU forms stream the same rows with the same per-wave loads)
                gv = [c for c in res if c[0] == "gemv"]
                if gv and N % 32 == 0:
                    ext = _native(x)
                    rr = torch.zeros(M, N, dtype=torch.bfloat16, device=dev)
                    sq = torch.empty(max_slots(N, M), M, dtype=torch.float32, device=dev)
                    for c in gv:
                        opts["gemv%d" % c[1]] = _time(lambda i: ext.gemv_resadd(x, ws[i % copies], rr, sq, c[1]))
                # small-batch MFMA GEMM with the epilogue fused (one launch), timed in its RESADD form
                # on the weight layout the fused ops stream (the panel copy where the model keeps one)
                if M <= SKE_MAX_M and N % 32 == 0 and K % 64 == 0:
                    rr = torch.zeros(M, N, dtype=torch.bfloat16, device=dev)
                    sq = torch.empty(max_slots(N, M), M, dtype=torch.float32, device=dev)
                    src = wps if wps is not None else ws
                    for sp in _SKE_SPLITS:
                        if sp > 1 and K // sp < 256:
                            continue
                        try:
                            opts["skE%d" % sp] = _time(lambda i: skinny_epi(x, src[i % copies], EPI_RESADD, sp, res=rr,
                                                                             ssq_out=sq))
                        except Exception:  # noqa: BLE001 - workspace / shape refused
                            pass
                if role is not None:
                    insitu = _retime_fused(tkey, role, opts, x, ws, wps, qkv_dims, dev, qkv_cache, wfs if M <= DG_MAX_M else None)
                    if insitu:
                        opts = insitu
                        if wfs is not None and M <= DG_MAX_M:
                            _P.frag_core[tkey] = _best_core(opts)
                _P.fused_core[tkey] = _best_core({c: t for c, t in opts.items() if not c.startswith("dg")})
                _P.fused_opts[tkey] = opts
            elif need_frag and tkey in _P.fused_core:
                _time_frag_core(tkey, role, x, ws, wps, qkv_dims, dev, qkv_cache, wfs)
            if verbose:
                bk = {k: min((c for c in res if c[0] == k), key=res.get, default=None)
                      for k in ("gemv", "skinny", "tg")}
                extra = " ".join(f"{k}={c[1:]}:{res[c]:.1f}us" for k, c in bk.items() if c)
                top = sorted(tgc, key=res.get)[:4]
                extra += " | tg top: " + " ".join(f"{c[1:]}:{res[c]:.1f}" for c in top)
                if post is not None:
                    extra += (f" | post {post:.1f}us | fused " +
                              " ".join(f"{k}:{v:.1f}" for k, v in _P.fused_opts[tkey].items()) +
                              f" -> core {_P.fused_core[tkey]}, with copies {_P.frag_core.get(tkey)}")
                print(f"gemm M={M} N={N} K={K} swiglu={sw}: best={best} {res[best]:.1f}us "
                      f"({N * K * 2 / res[best] / 1e3:.0f} GB/s, {2 * M * N * K / res[best] / 1e6:.0f} TF/s; "
                      f"blas {res[('blas',)]:.1f}us; {extra})", flush=True)
        del ws, wps, wfs


def plans() -> Dict:
    d = {str(k): v for k, v in _P.plans.items()}
    d.update({"tg" + str(k): v for k, v in _P.tg_plans.items()})
    d.update({"dg" + str(k): v for k, v in _P.dg_plans.items() if v})
    return d
