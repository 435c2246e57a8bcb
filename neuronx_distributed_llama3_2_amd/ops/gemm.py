"""GEMM entry points of the linear layers (csrc/gemm.cpp: hipBLASLt with per-shape autotuning).

`linear(x, w)` = x @ w^T, `matmul(a, b)` = a @ b, `wgrad_accumulate_(mg, go, x)` does
mg += go^T @ x with bf16 operands accumulating into the fp32 `main_grad` in place (one GEMM with
beta = 1, no bf16 temporary).  On CPU, or with NXD_TUNED_GEMM=0, they fall back to torch.
"""

from __future__ import annotations

import os
from typing import Optional

import torch

from ._ext import ext, gemm_ext, use_native

_ENABLED = os.environ.get("NXD_TUNED_GEMM", "1") == "1"


def set_overlap_safe(enabled: bool) -> None:
    """Select GEMM solutions without stream-K (csrc/gemm.cpp `no_streamk`): a persistent stream-K
    GEMM stalls while a concurrent collective holds one of its CUs.  Multi-rank training turns it
    on with NXD_GEMM_NO_STREAMK=1 (parallel_state.initialize_model_parallel)."""
    if not torch.cuda.is_available():
        return
    try:
        ext().gemm_set_no_streamk(1 if enabled else 0)
    except Exception:  # extension not built (CPU-only environments)
        pass


def _native(*t: torch.Tensor) -> bool:
    return _ENABLED and use_native(*t) and all(x.dtype in (torch.bfloat16, torch.float16) for x in t)


def linear(x: torch.Tensor, w: torch.Tensor, bias=None, out: torch.Tensor = None) -> torch.Tensor:
    """x [..., K] @ w[N, K]^T -> [..., N] (written into `out` if given: contiguous [..., N])."""
    shape = x.shape[:-1] + (w.shape[0],)
    if _native(x, w) and x.stride(-1) == 1:
        x2 = x.reshape(-1, x.shape[-1])
        y = out if out is not None else torch.empty(shape, dtype=x.dtype, device=x.device)
        gemm_ext().gemm(x2, w.t(), y.view(-1, w.shape[0]), None, 1.0, 0.0)
        return y + bias if bias is not None else y
    y = torch.nn.functional.linear(x, w, bias)
    if out is not None:
        out.copy_(y)
        return out
    return y


_ACTS = {"swiglu": 0, "relu2": 1}


def act_pays(rows: int, weight_rows: int, K: int, glu: bool = False) -> bool:
    """Whether csrc/act_gemm.hip takes a product and its activation, instead of a library product and the activation's own pass, which it was measured to be faster than: work for three quarters of the CUs (256 x 256
    results each), a reduction that the pass is not small beside, and rounds of the CUs that are filled to three quarters: what is left after whole rounds
    takes a whole one too, or, cut into 2 or 4 pieces, about two thirds of one (half of one if the pieces leave half of the CUs to themselves); up to a reduction of 1,024 the
    pass is so large a part that this does not matter (SwiGLU of 4,096 at 2,304 rows 53 / 43).  us, two launches / one,
    weights from memory: SwiGLU of 8,192 columns, reduction 2,048: 768 rows 52 / 47, 1,024 64 / 53, 1,664 110 / 94, 2,304 144 / 132, 4,096 226 / 197; of 14,336, 4,096: 512 rows
    108 / 94, 1,792 367 / 305, 5,120 977 / 799; of 11,008, 4,096: 4,096 681 / 507; squared ReLU of 12,288, 2,048: 640 rows 42 /
    42, 1,024 55 / 44, 4,096 178 / 145.  Rounds that are not filled (two launches): SwiGLU of 14,336, 4,096 at 384 rows 92 / 96, 640 146 / 157, 1,152 239 / 240, 8,192 at 1,152 85 /
    86, 3,072 at 1,280 121 / 126, 11,008 at 896 155 / 156, squared ReLU of 16,384, 4,096 at 1,280 150 / 156 (a part of a round below three quarters of it would pay in some places, which the rule
    leaves to two launches: 11,008 at 512 rows 93 / 82, squared ReLU of 12,288 at 896 50 / 44).  One line is older than the kernel is now: SwiGLU's reductions above 3,072 in four
    whole rounds and more went to two launches when a workgroup had one tile (706 / 714), and still do, though one would be the faster since it has up to four: of 14,336, 4,096 at
    4,096 / 12,288 rows 685 / 618, 2,047 / 1,886."""
    if K % 32 or K > 4096 or rows * weight_rows < 192 * 256 * 256:
        return False
    if K <= 1024:
        return True
    tiles = -(-rows // 256) * -(-weight_rows // 256)
    whole, tail = divmod(-(-tiles // 8), 32)   # of an XCD's CUs
    time = whole + (0 if tail == 0 else 0.45 if tail <= 4 else 0.67 if tail <= 16 else 1)
    return rows * weight_rows >= 0.75 * time * 256 ** 3 and not (glu and K > 3072 and tail == 0 and whole >= 4)


def linear_act(x: torch.Tensor, w: torch.Tensor, act: str) -> Optional[torch.Tensor]:
    """act(x [..., K] @ w^T) in one launch, or None where that is not done or not faster.  "swiglu": w [2 N, K] = [gate; up]; "relu2": w [N, K]."""
    K, N = w.shape[1], w.shape[0] // 2 if act == "swiglu" else w.shape[0]
    if not (_native(x, w) and x.dtype == w.dtype == torch.bfloat16 and act_pays(x.numel() // max(K, 1), w.shape[0], K, act == "swiglu")
            and N % (128 if act == "swiglu" else 8) == 0 and (N + 256) * K < 2 ** 31
            and x.shape[-1] == K and x.is_contiguous() and w.is_contiguous() and x.data_ptr() % 16 == 0 and w.data_ptr() % 16 == 0):
        return None
    y = torch.empty(x.shape[:-1] + (N,), dtype=x.dtype, device=x.device)
    gemm_ext().act_gemm(_ACTS[act], x.view(-1, K), w, y.view(-1, N))
    return y


def linear_f32(x: torch.Tensor, w: torch.Tensor, alpha: float = 1.0) -> torch.Tensor:
    """alpha * x [..., K] @ w[N, K]^T -> fp32 [..., N]: the accumulator unrounded (logits of 16-bit weights)."""
    if _native(x, w) and x.stride(-1) == 1:
        y = torch.empty(x.shape[:-1] + (w.shape[0],), dtype=torch.float32, device=x.device)
        gemm_ext().gemm(x.reshape(-1, x.shape[-1]), w.t(), y.view(-1, w.shape[0]), None, float(alpha), 0.0)
        return y
    y = torch.nn.functional.linear(x.float(), w.float())
    return y if alpha == 1.0 else y.mul_(alpha)


def matmul(a: torch.Tensor, b: torch.Tensor, out: torch.Tensor = None) -> torch.Tensor:
    """a [..., K] @ b [K, N] -> [..., N] (written into `out` if given: contiguous [..., N])."""
    shape = a.shape[:-1] + (b.shape[1],)
    if _native(a, b) and a.stride(-1) == 1:
        a2 = a.reshape(-1, a.shape[-1])
        y = out if out is not None else torch.empty(shape, dtype=a.dtype, device=a.device)
        gemm_ext().gemm(a2, b, y.view(-1, b.shape[1]), None, 1.0, 0.0)
        return y
    y = torch.matmul(a, b)
    if out is not None:
        out.copy_(y)
        return out
    return y


_WGRAD_BF16 = os.environ.get("NXD_WGRAD_BF16", "0") == "1"
_scratch = {}


# wgrad through transposed operands pays when the GEMM time saved beats the two transposes
# (~0.8e-12 * T*(N+K) s): measured, N*K/(N+K) above ~1200 -- Llama-3-8B gate_up, down, qkv and
# lm_head at TP=1; gate_up (975 -> 1116 TF/s), down (920 -> 944) and lm_head at TP=8, but not the
# TP=8 qkv / o shards (798 -> 566, 742 -> 440; profiles/r2_gemm_tp8_wgrad_layouts.jsonl).
# NXD_WGRAD_T=0 disables, =2 forces.
_WGRAD_T = os.environ.get("NXD_WGRAD_T", "1")


def _use_wgrad_t(go2: torch.Tensor, x2: torch.Tensor = None, K: int = None) -> bool:
    """TN layout for this wgrad?  x2 = None: the caller holds a contiguous token-major copy of x
    with K rows (only go2's strides matter)."""
    if _WGRAD_T == "0" or _WGRAD_BF16:
        return False
    T, N = go2.shape[0], go2.shape[1]
    K = x2.shape[1] if x2 is not None else K
    if T % 8 or N % 8 or K % 8 or go2.stride(-1) != 1 or go2.stride(0) % 8:
        return False
    if x2 is not None and (x2.stride(-1) != 1 or x2.stride(0) % 8):
        return False
    return _WGRAD_T == "2" or N * K / (N + K) > 1200


# Hand-written weight-gradient kernel (csrc/wgrad_gemm.hip): reads both token-major operands with
# the hardware transpose read and splits the token range over workgroups.  Measured against this
# module's hipBLASLt path (profiles/r3_wgrad_kernel_vs_hipblaslt.jsonl): faster on the skinny
# tensor-parallel shards -- TP=8 qkv 984 vs 743 TF/s, o 880 vs 717 (M*N/(M+N) < 1100) -- and
# 5-13 % slower than the bare TN GEMM on the large TP=1 shapes.  Counting the TN path's two operand
# transposes the isolated kernel should also win TP=1 qkv / o_proj, but inside the TP=1 step that
# routing measured +4.6 ms per 2 micro-batches (GEMM + wgrad kernel + transposes 531.9 vs 527.3 ms,
# profiles/r3_step_breakdown_wgrad_all_nocopy_rejected.txt), so `auto` keeps the skinny rule.  With
# the ping-pong main loop (profiles/r3_wgrad_pp_vs_hipblaslt.jsonl) the kernel also takes the
# vocabulary-sized output (lm_head) when no producer wrote a feature-major copy: TP=8 1201 vs 1074
# TF/s for the hipBLASLt path and its two transposes (the 1 GiB logits gradient), TP=1 a tie.
# NXD_WGRAD_KERNEL = auto | 1 (whenever the shapes allow) | 0.
#
# Token counts that are no multiple of 64 have no producer copies, and go to this kernel
# (unsplit from 128 tiles of 256 x 256 on: a second split's atomics cost more than the chip's idle part, 6,144 x 4,096 over 1,000
# tokens 88 us, in two splits 201, library 99) by how full its rounds of 256 tiles are.  Time of the library with its two
# transposes = 1: few tokens always (72: 0.39-0.89, 200: 0.50-0.92; 500, from 128 tiles on: 0.76-0.98); rounds three quarters full up
# to 1,000 (0.75-0.92; at 1,500 0.89-1.07), and from 7/8 at any even count (0.73-0.97 from 224 to 1,576 tiles up to 16,392
# tokens).  Less full: 128 tiles 1.13 over 1,000, 1.70 over 8,200; 280 tiles 1.22 over 3,000; 96 tiles 1.08 over 500.  Odd
# counts take no transposes: 0.83-0.95 at 1,001, 0.91-0.98 at 3,071, slower from 4,001 on.  M N / (M + N) measured up to 3,737.
# All of that with the main loop as it was; what fills its rounds comes here no more (wgrad_in_rounds).  With the loop as it is, time over the library's: ragged counts of 192 and
# 208 tiles 0.69-0.81 from 72 to 1,000 tokens, 128 tiles 0.81 up to 200 and 1.05 at 500, 264 and 280 tiles 0.86-0.94 up to 200 and 0.97 at 500, 96 tiles 0.87-0.93 up to 320, but 64
# tiles 1.3-1.6 there; vocabulary-sized ones in whole steps (16,032 to 128,256, 256 to 2,944 tokens) 0.79-0.95; M N / (M + N) < 1,100: 0.72-0.89 from 16,384 tokens on, 0.8-1.0
# at 8,192, and slower for fewer tokens (1.1-1.3 at 4,096, 1.4-1.7 at 512 to 2,048, 512 x 512 1.7-2.4): the line was drawn at 16,384 tokens of tensor-parallel
# shards, and has not been moved.  Nor have single rounds below seven eighths past 1,000 tokens (208 tiles, 3,001 tokens: 0.75).
_WG_KERNEL = os.environ.get("NXD_WGRAD_KERNEL", "auto")
_WG_SKINNY = 1100.0
_WG_WIDE = 16000
_WG_RAGGED = 4000.0
def _ragged_tokens(tiles: int, odd: bool) -> int:
    """Token counts (no multiple of 64) up to which a product of so many tiles goes to the wgrad kernel."""
    full = tiles / (256 * -(-tiles // 256))
    if tiles < 128:
        return 320
    return 512 if full < 0.75 else 1000 if full < 0.875 else 3072 if odd else 1 << 31


def _wgrad_kernel_splits(mg: torch.Tensor, go2: torch.Tensor, x2: torch.Tensor, has_copy: bool = False):
    """Token splits with which the wgrad kernel takes this product (0: its own choice), None: it does not."""
    if _WG_KERNEL == "0" or x2 is None or not _native(go2, x2) or mg.dtype != torch.float32:
        return None
    T, M = go2.shape
    N = x2.shape[1]
    if M % 8 or N % 8 or go2.stride(1) != 1 or x2.stride(1) != 1 or mg.stride(1) != 1:
        return None
    if go2.stride(0) % 8 or x2.stride(0) % 8 or go2.data_ptr() % 16 or x2.data_ptr() % 16:
        return None
    if T % 32 == 0 and (_WG_KERNEL == "1" or M * N / (M + N) < _WG_SKINNY or (not has_copy and max(M, N) >= _WG_WIDE)):
        return 0
    tiles = -(-M // 256) * -(-N // 256)
    if T % 64 and not has_copy and M * N / (M + N) < _WG_RAGGED and T <= _ragged_tokens(tiles, T % 8 != 0):
        return 1 if tiles >= 128 else 0
    return None


def _use_wgrad_kernel(mg: torch.Tensor, go2: torch.Tensor, x2: torch.Tensor, has_copy: bool = False) -> bool:
    return _wgrad_kernel_splits(mg, go2, x2, has_copy) is not None


# Whole steps of 64 tokens and no producer copy, M N / (M + N) < 2200: the wgrad kernel as well, with its own choice of splits.
# Its time over the library's (with two transposes from M N / (M + N) = 1,200 on), 64 to 16,384 tokens: 4,096 x 4,096 0.74-0.86,
# 2,048 x 8,192 0.69-0.85, 16,384 x 2,048 0.70-0.93, 3,584 x 4,096 0.77-0.90, 3,072 x 4,096 0.77-0.92; from 16,384 tokens on also smaller
# ones (2,048 x 2,048 0.76, 768 x 4,096 0.83).  The library is faster for few tiles over few tokens: 2,048 x 2,048 1.2-1.65 over 64 to 4,096
# tokens, 768 x 4,096 1.1-1.7, 512 x 512 1.1-2.4.  Time over that of the TN form of csrc/dense_gemm.hip, which was here before: 0.67-1.01.
# NXD_DENSE_WGRAD = auto | 1 (whenever the shapes allow) | 0.
_DENSE_WG = os.environ.get("NXD_DENSE_WGRAD", "auto")
_DENSE_WG_SKINNY = 2200.0


def _use_dense_wgrad(mg: torch.Tensor, go2: torch.Tensor, x2, has_copy: bool) -> bool:
    if _DENSE_WG == "0" or x2 is None or not _native(go2, x2) or mg.dtype != torch.float32:
        return False
    T, M = go2.shape
    N = x2.shape[1]
    if T % 64 or M % 8 or N % 8 or go2.stride(1) != 1 or x2.stride(1) != 1 or mg.stride(1) != 1:
        return False
    if go2.stride(0) % 8 or x2.stride(0) % 8 or mg.stride(0) % 4:
        return False
    if go2.data_ptr() % 16 or x2.data_ptr() % 16 or mg.data_ptr() % 16:
        return False
    return _DENSE_WG == "1" or (not has_copy and M * N / (M + N) < _DENSE_WG_SKINNY)


# Products of whole rounds of 256 tiles, or nearly: the wgrad kernel ahead of all the rules above and below, a producer's copy or not.  Its time over that of the
# library with its transposes (main loop with one read, address or load between two MFMAs, gradients from memory): counts that are no multiple of 64, 2,998 to
# 20,001 tokens: 256 tiles 0.72-0.81, 352 (two rounds, 0.69 full) 0.88-0.94, 384 0.87-0.94, 640 0.73-0.82, 768 0.71-0.80, 1,376 0.70-0.80, 2,000 0.74, 4,008 0.75; 1,000 to 1,501 of
# them: 352 0.83, 384 0.80-0.92, 640 0.80, 1,024 0.82, 4,096 0.69; 200: 4,096 0.75.  Whole steps of 64, 3,072 tokens: 384 0.95, 640 0.85, 688 0.85, 768 0.87, 896 0.92; 4,096 and
# 8,192: 352 0.93, 384 0.91-0.95, 400 0.86-0.89, 768 0.82-0.86, 1,376 0.76-0.78, 2,000 0.87.  Not: 512 to 2,048 tokens in whole steps (0.92-1.11), rounds that are less full (320 tiles
# 0.95-1.04 from 4,096 tokens on), one round below seven eighths.
_WG_WHOLE_TOKENS = 3072


def wgrad_in_rounds(T: int, M: int, N: int) -> bool:
    """Whether the weight gradient [M, N] of T tokens goes to the wgrad kernel because it fills its rounds of tiles: it reads both operands as they are, so
    nobody needs to write transposed copies for it."""
    tiles = -(-M // 256) * -(-N // 256)
    rounds = -(-tiles // 256)
    if _WG_KERNEL == "0" or _WGRAD_BF16 or _WGRAD_T == "2":   # (NXD_WGRAD_BF16=1, NXD_WGRAD_T=2: the library's products are asked for)
        return False
    if M % 8 or N % 8 or (T % 64 == 0 and T < _WG_WHOLE_TOKENS):
        return False
    return 8 * tiles >= 7 * 256 if rounds == 1 else 3 * tiles >= 2 * 256 * rounds


def _adds_in_rounds(mg: Optional[torch.Tensor]) -> bool:
    """Whether the wgrad kernel can add to this gradient a tile at a time."""
    return mg is not None and mg.dtype == torch.float32 and mg.dim() == 2 and mg.stride(1) == 1 and mg.stride(0) % 4 == 0 and mg.data_ptr() % 16 == 0


def kernel_gradients(*modules) -> bool:
    """Whether all these linear layers' weights have gradient buffers that the wgrad kernel adds to.  (16-bit buffers, and weights without one, are the library's, which
    wants a producer's transposed copies: an MLP forward and backward into 16-bit buffers, us with / without, 4,096 tokens, 4096 x 11008 2,856 / 2,893, 8,192, 4096 x 14336
    6,287 / 6,324.)"""
    return all(_adds_in_rounds(getattr(getattr(m, "weight", None), "main_grad", None)) for m in modules)


def _use_wgrad_in_rounds(mg: torch.Tensor, go2: torch.Tensor, x2) -> bool:
    if x2 is None or not _native(go2, x2) or go2.dtype != torch.bfloat16 or x2.dtype != torch.bfloat16 or not _adds_in_rounds(mg):
        return False
    if go2.stride(1) != 1 or x2.stride(1) != 1 or go2.stride(0) % 8 or x2.stride(0) % 8 or go2.data_ptr() % 16 or x2.data_ptr() % 16:
        return False
    return wgrad_in_rounds(go2.shape[0], go2.shape[1], x2.shape[1])


def _wgrad_scratch(n: int, dtype, device, tag: str = "") -> torch.Tensor:
    # one buffer per stream: the two halves of parallel_layers/stream_split.py transpose concurrently
    sid = torch.cuda.current_stream(device).stream_id if torch.device(device).type == "cuda" else 0
    key = (dtype, str(device), tag, sid)
    t = _scratch.get(key)
    if t is None or t.numel() < n:
        t = _scratch[key] = torch.empty(n, dtype=dtype, device=device)
    return t[:n]


def wgrad_accumulate_(mg: torch.Tensor, go2: torch.Tensor, x2, go_t: torch.Tensor = None,
                      x_t: torch.Tensor = None) -> None:
    """mg [N, K] (fp32) += go2[T, N]^T @ x2[T, K].

    `go_t` / `x_t`: optional contiguous [N, T] / [K, T] copies of go2 / x2 already written by their
    producers (the SwiGLU backward / forward), used instead of transposing when the TN layout is
    taken.  x2 may be None when only x_t was kept.

    Default: one hipBLASLt GEMM with fp32 C/D and beta = 1.  NXD_WGRAD_BF16=1: bf16-output GEMM
    into a reused scratch, then an fp32 add (the per-micro-batch weight gradient is rounded to
    bf16 before the fp32 accumulation — the precision of the reference's XLA matmul + fp32
    grad accumulation; hipBLASLt's bf16-output solutions run faster than its fp32-output ones)."""
    if go2.shape[0] == 0:
        return
    has_copy = go_t is not None or x_t is not None
    if _use_wgrad_in_rounds(mg, go2, x2) or _use_dense_wgrad(mg, go2, x2, has_copy):
        ext().wgrad_gemm(mg, go2, x2, 0, True)
        return
    splits = _wgrad_kernel_splits(mg, go2, x2, has_copy)
    if splits is not None:
        ext().wgrad_gemm(mg, go2, x2, splits, True)
        return
    if x_t is not None and not (x_t.dim() == 2 and x_t.is_contiguous() and x_t.shape[1] == go2.shape[0]):
        x_t = None
    if x2 is None and not (x_t is not None and _native(go2, x_t) and mg.is_contiguous()
                           and _use_wgrad_t(go2, K=x_t.shape[0])):
        x2 = x_t.t().contiguous()   # only the token-major copy was kept and the TN path is off
        x_t = None
    if x2 is None or (_native(go2, x2) and mg.is_contiguous()):
        if x2 is None or _use_wgrad_t(go2, x2):
            # T-contiguous operands: both transposed by the HIP kernel (~5 TB/s) into scratch, then
            # the TN GEMM (1.30-1.44 vs 1.06-1.16 PF/s on the NT layout, profiles/r2_gemm_layouts)
            T, N = go2.shape[0], go2.shape[1]
            K = x_t.shape[0] if x_t is not None else x2.shape[1]
            if go_t is not None and go_t.shape == (N, T) and go_t.is_contiguous() and go_t.dtype == go2.dtype:
                gt = go_t
            else:
                gt = transpose(go2, out=_wgrad_scratch(N * T, go2.dtype, go2.device, "gt").view(N, T))
            xt = x_t if x_t is not None else transpose(x2, out=_wgrad_scratch(K * T, x2.dtype, x2.device, "xt").view(K, T))
            ext().gemm(gt, xt.t(), mg, None, 1.0, 1.0)
            return
        if _WGRAD_BF16:
            tmp = _wgrad_scratch(mg.numel(), go2.dtype, go2.device).view(mg.shape)
            ext().gemm(go2.t(), x2, tmp, None, 1.0, 0.0)
            mg.add_(tmp)
            return
        ext().gemm(go2.t(), x2, mg, None, 1.0, 1.0)
        return
    if go2.is_cuda:
        torch.addmm(mg, go2.t(), x2, out_dtype=torch.float32, out=mg)
    else:
        mg.add_(go2.t().float().matmul(x2.float()))


# ----------------------------------------------------------------------------- dgrad layout
# hipBLASLt runs dX = dY W (W [N, K] row-major: the contraction dim is W's row dim) at 1.31-1.44
# PF/s on the Llama-3-8B shapes but at 1.56-1.69 PF/s when W is stored K-major (W^T [K, N]
# contiguous; profiles/r2_gemm_layouts.jsonl).  Training therefore keeps a K-major copy of every
# weight it back-propagates through, refreshed lazily by the first backward after the weights
# changed (one transpose per weight per optimizer step, HBM-bound, vs a faster dgrad in every
# micro-batch).  Staleness is detected by the optimizer's weight epoch (bumped by every optimizer
# step and checkpoint load that writes the weights outside autograd) plus the tensor's own
# version counter and storage pointer (any in-place torch write).  NXD_DGRAD_WT=0 disables it.
_DGRAD_WT = os.environ.get("NXD_DGRAD_WT", "1") == "1"
_weight_epoch = [0]


def weights_updated() -> None:
    """Tell the GEMM layer that weights were rewritten behind autograd's back (optimizer step)."""
    _weight_epoch[0] += 1


def transpose(src: torch.Tensor, out: torch.Tensor = None) -> torch.Tensor:
    """[R, C] -> contiguous [C, R] (HIP tiled transpose for bf16; torch elsewhere)."""
    dst = out if out is not None else torch.empty((src.shape[1], src.shape[0]), dtype=src.dtype, device=src.device)
    if use_native(src) and src.dtype == torch.bfloat16 and src.stride(-1) == 1 and src.shape[0] % 8 == 0 \
            and src.shape[1] % 8 == 0 and src.stride(0) % 8 == 0:
        ext().transpose_bf16(src, dst)
    else:
        dst.copy_(src.t())
    return dst


def _kmajor(weight: torch.Tensor) -> torch.Tensor:
    key = (_weight_epoch[0], weight._version, weight.data_ptr())
    wt = getattr(weight, "_nxd_wt", None)
    cur = torch.cuda.current_stream(weight.device)
    if wt is None or getattr(weight, "_nxd_wt_key", None) != key:
        if wt is None or wt.shape != (weight.shape[1], weight.shape[0]):
            wt = torch.empty((weight.shape[1], weight.shape[0]), dtype=weight.dtype, device=weight.device)
        transpose(weight.detach(), out=wt)
        weight._nxd_wt = wt
        weight._nxd_wt_key = key
        weight._nxd_wt_ev = torch.cuda.Event()
        weight._nxd_wt_ev.record(cur)
        weight._nxd_wt_stream = cur.stream_id
    elif getattr(weight, "_nxd_wt_stream", cur.stream_id) != cur.stream_id:
        # written on another stream (the other half of stream_split): wait for the transpose
        cur.wait_event(weight._nxd_wt_ev)
        wt.record_stream(cur)
    return wt


def dgrad(go: torch.Tensor, weight: torch.Tensor, out: torch.Tensor = None) -> torch.Tensor:
    """dX = go [..., N] @ weight [N, K] -> [..., K] (the input gradient of y = x W^T)."""
    if _DGRAD_WT and _native(go, weight) and go.stride(-1) == 1 and weight.dim() == 2 and weight.shape[0] % 8 == 0 \
            and weight.shape[1] % 8 == 0 and weight.is_contiguous():
        wt = _kmajor(weight)
        return matmul(go, wt.t(), out=out)
    return matmul(go, weight, out=out)
