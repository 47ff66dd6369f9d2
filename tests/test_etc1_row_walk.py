"""The ETC1 encoder scores a row of intensity modifiers by one general walk for
every lane; rg_etc1 (evaluate_solution_fast, rg_etc1.cpp:1767-1885) has
shortcuts for rows that lie wholly above or below the sub-block's lumas and
leaves some rows out early.  Both restated in numpy must choose the same row,
selectors and error; all integers, so exactly.
This argues the walk only: the kernel itself is held against the oracle on the
GPU in tests/test_etc1_gpu.py."""
import numpy as np
import pytest

ROWS = np.array([[-8, -2, 2, 8], [-17, -5, 5, 17], [-29, -9, 9, 29], [-42, -13, 13, 42],
                 [-60, -18, 18, 60], [-80, -24, 24, 80], [-106, -33, 33, 106],
                 [-183, -47, 47, 183]])


def reference_walk(px, base):
    luma = px.sum(1)
    order = np.argsort(luma, kind="stable")
    lo, hi = luma[order[0]], luma[order[7]]
    best = (1 << 62, 0, None)
    for row in range(7, -1, -1):
        c = np.clip(base + ROWS[row][:, None], 0, 255)
        y = c.sum(1)
        mid = y[:3] + y[1:]
        if 2 * hi < mid[0]:
            if y[0] > hi and y[0] - hi >= best[0]:
                continue
            sel = np.zeros(8, int)
        elif 2 * lo >= mid[2]:
            if lo > y[3] and lo - y[3] >= best[0]:
                continue
            sel = np.full(8, 3)
        else:
            sel, cur = np.zeros(8, int), 0
            for i in order:
                while cur < 3 and 2 * luma[i] >= mid[cur]:
                    cur += 1
                sel[i] = cur
        total = int(((px - c[sel]) ** 2).sum())
        if total < best[0]:
            best = (total, row, sel)
            if not total:
                break
    return best


def general_walk(px, base):
    luma2 = 2 * px.sum(1)
    norm = int((px * px).sum())
    best = (1 << 62, 0, None)
    for row in range(7, -1, -1):
        c = np.clip(base + ROWS[row][:, None], 0, 255)
        y = c.sum(1)
        mid = y[:3] + y[1:]
        sel = np.where(luma2 >= mid[2], 3,
                       np.where(luma2 >= mid[1], 2, np.where(luma2 >= mid[0], 1, 0)))
        e = np.concatenate([c[sel], 64 * sel[:, None]], 1)  # the index rides in the top byte
        idx2 = int((sel & 1).sum() + 4 * (sel >> 1).sum() + 4 * (sel == 3).sum())
        total = norm - 2 * int((px * e[:, :3]).sum()) + int((e * e).sum()) - (idx2 << 12)
        if total < best[0]:
            best = (total, row, sel)
    return best


@pytest.mark.parametrize("spread", [1, 8, 40, 256])
def test_general_walk_equals_the_reference_shortcuts(spread):
    rng = np.random.default_rng(spread)
    for _ in range(600):
        centre = rng.integers(0, 256, 3)
        px = np.clip(centre + rng.integers(-spread, spread, (8, 3)), 0, 255)
        base = np.clip(centre + rng.integers(-spread - 4, spread + 4, 3), 0, 255)
        a, b = reference_walk(px, base), general_walk(px, base)
        assert a[:2] == b[:2] and np.array_equal(a[2], b[2])
