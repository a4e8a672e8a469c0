"""Host-side check of the forward kernels' workgroup -> query-block mapping.

The forwards (``csrc/fwd_common.hpp``, ``tile_coords_lpt``) deal workgroups to
XCDs round-robin and give each XCD a contiguous run of query blocks, total // 8
of them and one more for the first total % 8 XCDs. Inside each window of 8192
query tokens of a run (64 dispatches at block 128, 128 at block 64; the last
window spans up to two of them) the query blocks are taken longest first, ties
by index: the workgroup at place r selects the r-th largest key (exact-block
count, then earlier index first), built bit by bit from ballots. The mapping
must be a permutation of ``[0, grid)`` for every grid size and every count
pattern, or a query block is computed twice and another never (or an index
leaves the buffers). This restates the kernel's arithmetic and checks the
permutation and the order, which the kernel's parity tests only see for the
grid sizes they run.
"""
import numpy as np
import pytest


def _select(counts, WINDOW, NT):
    """The kernel's selection, one entry per workgroup: keys are unique (count
    clamped to [0, NT], earlier index first)."""
    total, idx = len(counts), 2 * WINDOW
    bits = idx.bit_length() - 1
    out = np.empty(total, dtype=np.int64)
    for w in range(total):
        x, li, q8, rem = w & 7, w >> 3, total >> 3, total & 7
        per = q8 + (x < rem)
        tail0 = (per - 1 - WINDOW) & ~(WINDOW - 1) if per > WINDOW else 0
        win0 = min(li & ~(WINDOW - 1), tail0)
        base, r = x * q8 + min(x, rem) + win0, li - win0
        nwin = per - win0 if win0 == tail0 else WINDOW
        assert 0 <= r < nwin <= idx and 0 <= base and base + nwin <= total
        key = [(min(max(counts[base + i], 0), NT) << bits) | (idx - 1 - i) for i in range(nwin)]
        sel = 0
        for bit in range(NT.bit_length() - 1 + bits, -1, -1):
            if sum(k >= sel | (1 << bit) for k in key) > r:
                sel |= 1 << bit
        out[w] = base + idx - 1 - (sel & (idx - 1))
    return out


def _windows(per, WINDOW):
    """The windows of a run of `per` query blocks, as (first, size): whole ones while
    more than two windows' worth would be left, then what is left in one."""
    first, out = 0, []
    while per - first > 2 * WINDOW:
        out.append((first, WINDOW))
        first += WINDOW
    return out + [(first, per - first)]


TOTALS = [1, 7, 8, 9, 24, 65, 513, 8 * 64, 8 * 65 + 3, 8 * 128, 8 * 128 + 8, 8 * 129 + 5, 8 * 192, 2056, 3079]


@pytest.mark.parametrize("total", TOTALS)
@pytest.mark.parametrize("window", [64, 128])
def test_dispatch_map_is_permutation(total, window):
    """For any counts (ties, negative and beyond NT too) and any grid."""
    rng = np.random.default_rng(total + window)
    for lo, hi in ((0, 5), (-2, 12)):
        counts = rng.integers(lo, hi, size=total).tolist()
        assert sorted(_select(counts, window, 8).tolist()) == list(range(total))


@pytest.mark.parametrize("total", TOTALS)
@pytest.mark.parametrize("window", [64, 128])
def test_dispatch_map_longest_first_within_window(total, window):
    """Counts descend, ties by index, along the dispatches of every window of every
    XCD's run, the last one and runs of unequal length among them."""
    rng = np.random.default_rng(3 * total + window)
    counts = rng.integers(0, 9, size=total)
    m = _select(counts.tolist(), window, 8)
    start = 0
    for xcd in range(min(8, total)):
        run = m[xcd::8]
        for first, size in _windows(len(run), window):
            blocks = np.arange(start + first, start + first + size)
            order = blocks[np.argsort(-counts[blocks], kind="stable")]
            assert np.array_equal(run[first:first + size], order)
        start += len(run)
    assert start == total
