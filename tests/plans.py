"""The sizes at which the decode step writes key lists, restated from the rule in csrc/select.h (fused_tiling, list_plan) so
that a test can say which select its shapes reach. test_abi.py holds these against the library's own sizes."""
from __future__ import annotations

import math

import numpy as np


def align(x, n=256):
    return (x + n - 1) // n * n


def fused_tiling(BG, lo, hi):
    """(sub-tiles of 512 columns per score workgroup, workgroups per row)"""
    span = ((hi + 7) & ~7) - (lo & ~7)
    blocks = BG * ((span + 511) // 512)
    nsub = 8 if blocks >= 8 * 256 else 4 if blocks >= 4 * 256 else 2 if blocks >= 2 * 256 else 1
    return nsub, (span + 512 * nsub - 1) // (512 * nsub)


def list_plan(BG, lo, hi, k, max_m=131072):
    """(lmin, cap) of a key list: the keys it holds at least, and its entries (0, 0: no lists at this shape). max_m: 131072
    where the row list stays in the step, else 32768."""
    M = hi - lo
    if k <= 0 or M <= 0 or M > max_m:
        return 0, 0
    nsub, tiles = fused_tiling(BG, lo, hi)
    n = 512 * nsub
    share = (k * n + M - 1) // M
    lmin = share + 3 * math.isqrt(share) + 16
    return (0, 0) if tiles > 128 or 2 * lmin > n else (lmin, min(n, (lmin + 192 + 63) // 64 * 64))


def list_cap(BG, lo, hi, k, max_m=131072):
    return list_plan(BG, lo, hi, k, max_m)[1]


def list_bytes(BG, lo, hi, k, max_m=131072):
    cap = list_cap(BG, lo, hi, k, max_m)
    tiles = fused_tiling(BG, lo, hi)[1] if cap else 0
    return align(BG * tiles * cap * 8) + align(BG * tiles * 8)


def head_groups(BG, h, P):
    """Head groups of the one-launch select and attend: powers of two dividing h while the grid stays within 256."""
    Q = 1
    while h % (2 * Q) == 0 and BG * P * 2 * Q <= 256:
        Q *= 2
    return Q


def one_launch(BG, lo, hi, legal, k, h, P):
    """Whether a step of r = 32 over an aligned table, whose row list stays in the call, selects and attends in one launch."""
    if h * 128 > 512 or list_cap(BG, lo, hi, k) == 0:
        return False
    S = lo + (legal - hi) + k
    return h // head_groups(BG, h, P) in (1, 2, 4) and -(-S // P) <= (8192 if hi - lo > 32768 else 4096)


def score_keys(scores):
    """The order-preserving 32-bit key of float32 scores without NaN (-0.0 as +0.0)."""
    bits = (np.asarray(scores, dtype=np.float32) + np.float32(0.0)).view(np.uint32)
    return np.where(bits >> 31, ~bits, bits | np.uint32(0x80000000))


def list_paths(scores, BG, lo, hi, k):
    """How the list select reads one row of scores [M]: (tiles recomputed from the table, tiles read from their stored keys,
    keys that share the threshold's first digit, those that share its first two)."""
    nsub, tiles = fused_tiling(BG, lo, hi)
    lmin, cap = list_plan(BG, lo, hi, k)
    key = score_keys(scores)
    kth = np.sort(key)[-k]
    b1 = kth >> 21
    list_of = ((np.arange(lo, hi) - (lo & ~7)) // 512) % tiles
    recomputed = stored = 0
    for w in range(tiles):
        d = np.sort(key[list_of == w] >> 21)[::-1]
        if d.size == 0:
            continue
        least = d[min(lmin, d.size) - 1] if d.size >= lmin else 0
        length = int((d >= least).sum())
        stored += length > cap
        recomputed += length <= cap and least > b1
    return recomputed, stored, int((key >> 21 == b1).sum()), int((key >> 10 == kth >> 10).sum())
