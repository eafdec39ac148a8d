"""The sizes at which the decode step writes key lists, restated from the rule in csrc/select.h (fused_tiling, list_plan) so
that a test can say which select its shapes reach. test_abi.py holds these against the library's own sizes."""
from __future__ import annotations

import math


def align(x, n=256):
    return (x + n - 1) // n * n


def fused_tiling(BG, lo, hi):
    """(sub-tiles of 512 columns per score workgroup, workgroups per row)"""
    span = ((hi + 7) & ~7) - (lo & ~7)
    blocks = BG * ((span + 511) // 512)
    nsub = 8 if blocks >= 8 * 256 else 4 if blocks >= 4 * 256 else 2 if blocks >= 2 * 256 else 1
    return nsub, (span + 512 * nsub - 1) // (512 * nsub)


def list_cap(BG, lo, hi, k, max_m=131072):
    """Entries of a key list (0: no lists at this shape). max_m: 131072 where the row list stays in the step, else 32768."""
    M = hi - lo
    if k <= 0 or M <= 0 or M > max_m:
        return 0
    nsub, tiles = fused_tiling(BG, lo, hi)
    n = 512 * nsub
    share = (k * n + M - 1) // M
    lmin = share + 3 * math.isqrt(share) + 16
    return 0 if tiles > 128 or 2 * lmin > n else min(n, (lmin + 192 + 63) // 64 * 64)


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
