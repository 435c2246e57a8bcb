"""Decode-path linear ops (csrc/few_rows.hip, gemv.hip): skinny GEMM for M <= 32 tokens (8 with a bias) with bf16 or int8
weights, optional per-row / per-tensor scale, bias and fused SwiGLU epilogue; int8 -> bf16 dequantisation
for the prefill path.  CPU / large-M calls fall back to dequantise + GEMM."""

from __future__ import annotations

from typing import Optional

import torch

from ._ext import ext, use_native
from .gemm import linear as _linear, linear_act


def dequantize_weight(w: torch.Tensor, scale: Optional[torch.Tensor], dtype=torch.bfloat16) -> torch.Tensor:
    """int8 [N, K] (* scale [N] / [N,1] / [1]) -> dtype [N, K]; bf16 weights pass through."""
    if w.dtype != torch.int8:
        return w
    if use_native(w) and dtype == torch.bfloat16 and w.shape[1] % 16 == 0:
        s = scale.reshape(-1).float().contiguous() if scale is not None else None
        out = torch.empty(w.shape, dtype=torch.bfloat16, device=w.device)
        if s is not None and s.numel() == 1:
            ext().dequant_int8(w, s.expand(w.shape[0]).contiguous(), 1.0, out)
        else:
            ext().dequant_int8(w, s, 1.0, out)
        return out
    if scale is None:
        s = 1.0
    elif scale.numel() == 1:
        s = scale.float().reshape(())
    else:
        s = scale.float().reshape(-1, 1)
    return (w.float() * s).to(dtype)


def few_rows_pay(rows: int, weight_rows: int, K: int, fused: bool = False) -> bool:
    """Whether a bf16 product of up to 32 rows is faster in csrc/few_rows.hip than in the library's product.  fused: with
    an element-wise epilogue (SwiGLU, squared ReLU), which the library follows with a launch.

    Up to 8 rows always (the library's time is that of 16).  Up to K = 4,224 the kernel keeps the activations in registers:
    9 to 16 rows take 0.42-1.01 of the library's time over 256 to 128,256 weight rows; 17 to 32 rows 0.43-1.04 up to K = 2,048.
    Beyond it (K 2,304 to 4,096): up to 3,072 weight rows 0.39-0.95 at 17 to 32 rows (2,048 x 4,096 at 32 8.4 us, library 12-18);
    4,096 0.54-0.94 up to 20 rows and 0.58-1.03 at 24, at 25 to 32 0.60-0.82 up to K = 3,072 and 0.98-1.09 at 4,096; from 12,288 on 0.74-0.98 up to
    24 rows (0.83-1.02 at more from K = 3,072 on, 12,288 x 4,096 at 32 22.5 us, library 25.7; 0.92-1.12 at K = 2,304); between, 0.91-1.16
    and mostly above 1 (at K = 2,304 0.52-1.30).  Longer reductions read them once per workgroup: 8,192 x 10,240 at 9 / 16 / 32 rows 33.9 /
    40.1 / 56.4 us, library 34.8 / 35.6 / 37.4."""
    if rows <= 8:
        return True
    if K > 4224:
        return False
    if rows <= 16 or K <= 2048 or fused or weight_rows >= 16384:
        return True
    if weight_rows >= 12288:
        return rows <= 24 or K >= 3072
    return weight_rows <= (4096 if rows <= 24 or K <= 3072 else 3072)


def skinny_linear(x: torch.Tensor, w: torch.Tensor, scale: Optional[torch.Tensor] = None,
                  bias: Optional[torch.Tensor] = None, glu: bool = False) -> torch.Tensor:
    """x [..., K] @ W^T (+ bias) (W bf16 or int8 [Nw, K]); glu=True: W = [gate; up] rows and the
    result is silu(gate) * up of width Nw / 2."""
    K = x.shape[-1]
    lead = x.shape[:-1]
    M = x.numel() // K
    Nw = w.shape[0]
    N = Nw // 2 if glu else Nw
    # what csrc/few_rows.hip takes, up to 32 rows: int8 with a scale or bf16 without, no bias, weights under 2 GB at 32-bit
    # offsets (rows of a strided weight lie further apart than numel says)
    # (int8: the other way is to widen the weights in memory first, 2 to 5 times slower)
    few = (bias is None and w.dtype == (torch.bfloat16 if scale is None else torch.int8) and N > 0
           and (w.dtype == torch.int8 or few_rows_pay(M, Nw, K, glu)) and w.numel() * w.element_size() < 2 ** 31 and (Nw + 16) * w.stride(0) * w.element_size() < 2 ** 32)
    if use_native(x, w) and M <= (32 if few else 8) and x.dtype == torch.bfloat16 and w.stride(-1) == 1:
        x2 = x.reshape(M, K)
        if x2.stride(1) != 1 or x2.stride(0) % 8 or x2.stride(0) >= 2 ** 24 or x2.data_ptr() % 16:
            x2 = x2.contiguous()
        epl = 16 if w.dtype == torch.int8 else 8
        if K % epl == 0 and w.data_ptr() % 16 == 0 and w.stride(0) % epl == 0:
            y = torch.empty((M, N), dtype=torch.bfloat16, device=x.device)
            s = None
            if scale is not None:
                s = scale.reshape(-1).float()
                s = (s.expand(Nw) if s.numel() == 1 else s).contiguous()
            ext().gemv(x2, w, s, 1.0, bias, y, glu)
            return y.view(lead + (N,))
    wd = dequantize_weight(w, scale, x.dtype) if w.dtype == torch.int8 else w
    if glu and bias is None:
        y = linear_act(x, wd, "swiglu")
        if y is not None:
            return y
    y = _linear(x, wd, bias)
    if glu:
        from .activations import swiglu

        y = swiglu(y)
    return y


def expert_linear(x: torch.Tensor, w_t: torch.Tensor, eidx: torch.Tensor, xdiv: int = 1,
                  glu: bool = False) -> torch.Tensor:
    """MoE decode projection for P (token, expert-slot) pairs: y[p] = x[p // xdiv] @ W[eidx[p]]^T,
    W given output-major as w_t [E, Nw, K]; glu=True: rows [gate; up] -> silu(gate) * up.  Reads
    only the selected experts' weights (csrc/gemv.hip expert mode); static shapes, no host sync,
    so it is captured in the decode hipGraph."""
    P = eidx.numel()
    Nw, K = w_t.shape[1], w_t.shape[2]
    N = Nw // 2 if glu else Nw
    if use_native(x, w_t) and x.dtype == torch.bfloat16 and w_t.dtype == torch.bfloat16 and w_t.stride(2) == 1 \
            and K % 8 == 0 and w_t.stride(1) % 8 == 0 and w_t.stride(0) % 8 == 0 and w_t.data_ptr() % 16 == 0:
        x2 = x.reshape(-1, K)
        if x2.stride(1) != 1 or x2.stride(0) % 8 or x2.data_ptr() % 16:
            x2 = x2.contiguous()
        y = torch.empty((P, N), dtype=torch.bfloat16, device=x.device)
        ext().expert_gemv(x2, w_t, eidx.reshape(-1).to(torch.int32).contiguous(), int(xdiv), y, glu)
        return y
    rows = x.reshape(-1, K).index_select(0, torch.arange(P, device=x.device) // xdiv)
    y = torch.bmm(rows.unsqueeze(1), w_t.index_select(0, eidx.reshape(-1).long()).transpose(1, 2)).squeeze(1)
    if glu:
        from .activations import swiglu

        y = swiglu(y)
    return y
