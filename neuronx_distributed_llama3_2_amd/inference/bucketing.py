"""Sequence-length bucketing (reference: examples/inference/modules/autobucketing.py:6-126).

Buckets are powers of two from the minimum up to (and including) the maximum length.  Prompts are
right-padded to the smallest bucket that holds the longest prompt of the batch (`prefill_lengths`: or
to halfway between two of them, for batches of 1,024 tokens and more) so the context encoder sees a
handful of distinct shapes (stable allocator pools, reusable GEMM heuristics); the decode path needs
no length buckets because attention reads the KV cache up to a per-sequence device-side length.
"""

from __future__ import annotations

from math import log2
from typing import List, Sequence

import torch


def generate_buckets(min_length: int, max_length: int) -> List[int]:
    if min_length >= max_length:
        return [max_length]
    lo = int(log2(min_length))
    hi = round(log2(max_length))
    return [2 ** i for i in range(lo, hi)] + [max_length]


def select_bucket(length: int, buckets: Sequence[int]) -> int:
    for b in sorted(buckets):
        if length <= b:
            return b
    raise ValueError(f"length {length} exceeds the largest bucket {max(buckets)}")


# Tokens of a padded batch from which on a length halfway between two buckets pays: below, the weights' bytes bound the prefill and a
# quarter fewer tokens take little off (Llama-3.2-1B, 1 x 512 -> 1 x 384 tokens 2.22 -> 2.10 ms; 1 x 1,024 -> 768 3.12 -> 2.65, 3 x 1,024 -> 768
# 6.31 -> 5.34, 1 x 2,048 -> 1,536 4.98 -> 4.09), while each length costs its graph's capture once
# (0.2 s, in the first request that needs it: no length is captured ahead).
HALFWAY_TOKENS = 1024


def generated(config) -> bool:
    """Whether the configuration's buckets are the generated ones."""
    top = getattr(config, "max_context_length", 0)
    return bool(getattr(config, "buckets_generated", False) and top and list(config.buckets) == generate_buckets(min(128, top), top))


def prefill_lengths(config, batch: int, halfway: bool = True) -> List[int]:
    """Lengths that prompts of a batch are padded to: the configuration's buckets and its maximum length, and where the buckets are
    the generated ones (a caller's own list stands as it is) and `halfway` lengths may be used 1.5 times every bucket whose next one
    holds HALFWAY_TOKENS in the batch."""
    lengths = list(config.buckets)
    if halfway and generated(config):
        lengths += [lo * 3 // 2 for lo, hi in zip(lengths, lengths[1:]) if lo >= 128 and batch * hi >= HALFWAY_TOKENS and lo * 3 // 2 < hi]
    return lengths + [config.max_length]


def packed_rows(total: int) -> int:
    """Rows that `total` tokens of a batch are given where they lie one after the other: multiples of an eighth of the power of two below, of
    128 at least: eight for twice the tokens.  The library's products are tuned for each once (45 ms of a process, Llama-3.2-1B)."""
    step = max(128, (1 << (total - 1).bit_length()) // 16)
    return -(-total // step) * step


# Packed keys (batch, padded length, rows) that an application keeps, with their graphs where they have come often enough: one batch size and padded length alone
# has 11 (3 x 768), 24 (8 x 1,024) or 42 (32 x 2,048) row counts for which packing pays.
PACKED_KEYS = 64


def packing_pays(rows: int, batch: int, length: int) -> bool:
    """Whether prompts are encoded without their padding, in so many rows instead of `batch` times `length`: an eighth fewer, which is more than reading the
    lengths on the host costs (50 us of 3 to 10 ms)."""
    return batch * length >= HALFWAY_TOKENS and 8 * rows <= 7 * batch * length


def pad_to_bucket(input_ids: torch.Tensor, attention_mask: torch.Tensor, buckets: Sequence[int], pad_token: int):
    """Right-pad [B, T] ids / mask to the selected bucket length."""
    T = input_ids.shape[1]
    b = select_bucket(T, buckets)
    if b == T:
        return input_ids, attention_mask
    pad = b - T
    ids = torch.nn.functional.pad(input_ids, (0, pad), value=pad_token)
    mask = torch.nn.functional.pad(attention_mask, (0, pad), value=0)
    return ids, mask
