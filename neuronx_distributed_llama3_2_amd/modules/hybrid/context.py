"""What a mixer needs to know about the step it runs in."""

from __future__ import annotations

from dataclasses import dataclass
from typing import Optional

import torch

from ...ops.gemv import few_rows_pay


@dataclass
class StepContext:
    """T new tokens for each of B sequences (row b * T + t of every activation).  positions: int64, the
    first new token's in column 0; lengths [B] int32: valid new tokens (None: all T); slots [B] int32
    cache slots (None: 0..B-1); prompt: every sequence starts at position 0 in this step."""

    B: int
    T: int
    positions: torch.Tensor
    lengths: Optional[torch.Tensor]
    slots: Optional[torch.Tensor]
    prompt: bool
    fused: bool = True
    tickets: Optional[torch.Tensor] = None   # of ops.linear_few, for steps of few rows


# rows of a fused projection are padded to this, so that every row of its output is 16-byte aligned
ROW_ALIGN = 16


def padded_rows(n: int) -> int:
    return (n + ROW_ALIGN - 1) // ROW_ALIGN * ROW_ALIGN


# rows up to which a projection is a dot product a wave (csrc/hybrid/gemv_hyper.hip), and up to which it is
# a matrix-core product that streams the weights (csrc/few_rows.hip, some in csrc/hybrid/expert_decode.hip)
FEW_ROWS, SOME_ROWS = 2, 32


def few_rows(x: torch.Tensor, w: torch.Tensor, limit: int = FEW_ROWS) -> bool:
    return x.is_cuda and x.shape[0] <= limit and x.dtype == w.dtype == torch.bfloat16 and w.shape[1] % 8 == 0 and x.is_contiguous()


def streams(rows: int, weight_rows: int, K: int, fused: bool) -> bool:
    """Whether ops.linear_few is the faster product of up to SOME_ROWS rows.  Up to 16 rows it has the faster of two kernels;
    with more, long reductions are split (up to 8,192 weight rows: 0.45-1.18 of the library's time, mostly below 1;
    12,288 x 8,192 unsplit at 32 rows 57 us, library 47)."""
    if rows <= 16:
        return True
    return weight_rows <= 8192 if K > 4224 else few_rows_pay(rows, weight_rows, K, fused)


def linear(x: torch.Tensor, mod: torch.nn.Module, fused: bool = False, epilogue: str = "store",
           tickets: Optional[torch.Tensor] = None) -> torch.Tensor:
    """x [M, K] @ mod.weight^T: through the module's packed copy when the layout pass chose it; fused: a few
    rows by the kernels that stream the weights.  epilogue "relu2": its squared ReLU."""
    from ... import ops
    from ...trace.weight_layout import packed_linear, packed_linear_act

    if fused and few_rows(x, mod.weight, SOME_ROWS) and streams(x.shape[0], *mod.weight.shape, epilogue != "store"):
        if x.shape[0] <= FEW_ROWS:
            return ops.decode_linear(mod.weight, x, epilogue=epilogue)
        return ops.linear_few(x, mod.weight, epilogue, tickets=tickets)
    return packed_linear_act(mod, x, mod.weight, None, "relu2") if epilogue == "relu2" else packed_linear(mod, x, mod.weight)


def step_tickets(rows: int, device) -> Optional[torch.Tensor]:
    """Zeroed counters for the projections of a step of so many rows."""
    from ...ops.experts import LINEAR_TICKETS

    if torch.device(device).type != "cuda" or not FEW_ROWS < rows <= SOME_ROWS:
        return None
    return torch.zeros(LINEAR_TICKETS, dtype=torch.int32, device=device)


def small(*shape, device=None) -> torch.nn.Parameter:
    """A small parameter that enters 32-bit computations: kept in fp32 whatever the model's dtype."""
    return torch.nn.Parameter(torch.empty(*shape, dtype=torch.float32, device=device), requires_grad=False)
