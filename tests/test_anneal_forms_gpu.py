"""The annealing's forms (one lane per pixel for small lists, one lane per
candidate with a handed-over tail for large ones) and the set-up's (one launch
or one per mode) at the sizes where the choice changes, for every search that
takes them: whole images against the oracle, and large jobs against the same
blocks encoded in smaller ones."""
import ctypes
import os

import numpy as np
import pytest

from fastc_amd import synth
from tests.test_selection import random_selections

pytestmark = pytest.mark.gpu
WEIGHTS = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                       "fastc_amd", "data", "bc7_ranker.npy")


def _diff(a, b):
    return np.nonzero((a.reshape(-1, 16) != b.reshape(-1, 16)).any(axis=1))[0]


@pytest.mark.parametrize("w,h,q", [(512, 512, 4), (516, 512, 4), (8, 4, 4), (400, 400, 4),
                                   (512, 512, 16)])
def test_reference_search_matches_oracle(fh, oracle, w, h, q):
    """16384 blocks (the last size where the list's length chooses the form:
    one lane per candidate at quality 4, one per pixel at 16), 16512 (one lane
    per candidate always), 10000 (one per pixel, with the choice) and two,
    with the work counts."""
    img = synth.generate(w, h, 31)
    print(f"anneal forms {w}x{h} q={q}", flush=True)
    L = oracle.lib()
    L.ora_anneal_point_count(1)
    ref, ref_wm = oracle.bc7_compress(img, quality=q, seed=9, q0_guard=True)
    want = L.ora_anneal_point_count(1)
    wm = ctypes.c_uint32(0xFFFFFFFF)
    fh.set_work_counting(True)
    try:
        got = fh.compress(img, quality=q, seed=9, wm_counter=wm)
        n_ref, n_gpu = fh.work_counts()
    finally:
        fh.set_work_counting(False)
    bad = _diff(got, ref)
    assert bad.size == 0, f"{bad.size} blocks differ, first {bad[:8]}"
    assert wm.value == ref_wm
    assert n_ref == want and n_gpu % 16 == 0 and n_gpu >= n_ref
    plain = fh.compress(img, quality=q, seed=9, wm_counter=ctypes.c_uint32(0xFFFFFFFF))
    assert np.array_equal(plain, got)


@pytest.mark.parametrize("w,h,q", [(512, 512, 0), (516, 512, 2)])
def test_nonuniform_metric_matches_oracle(fh, oracle, w, h, q):
    """The nonuniform metric on the last size of the merged set-up and, with
    annealing, the first of one launch per mode: the waves' steps for one,
    two and three subsets."""
    img = synth.generate(w, h, 12)
    print(f"nonuniform forms {w}x{h}", flush=True)
    ref, ref_wm = oracle.bc7_compress(img, quality=q, seed=4, q0_guard=True, metric=1)
    wm = ctypes.c_uint32(0xFFFFFFFF)
    got = fh.compress(img, quality=q, seed=4, wm_counter=wm, metric=1)
    bad = _diff(got, ref)
    assert bad.size == 0, f"{bad.size} blocks differ, first {bad[:8]}"
    assert wm.value == ref_wm


def _row_rects(side, parts):
    """The image's rows in equal parts: (rect, first row, rows) of each."""
    rows = side // parts
    for k in range(parts):
        y0, y1 = k * rows, (k + 1) * rows
        # up to the start of the next part's first row
        yield ((0, y0, 0, y1) if y1 < side else (0, y0, side, side)), y0, rows


@pytest.mark.parametrize("search", ["nonuniform", "statistics", "selections"])
def test_other_searches_compose(fh, search):
    """25600 blocks, annealed, equal their quarters (which run the forms for
    small jobs, held against the oracle in those searches' own tests)."""
    side, parts = 640, 4
    img = synth.generate(side, side, 23)
    n = (side // 4) ** 2
    sels = None
    if search == "selections":
        sels = np.tile(random_selections(256, 3, 12), n // 256)
    print(f"anneal forms {search}", flush=True)

    def encode(rect, first, count):
        wm = ctypes.c_uint32(0xFFFFFFFF)
        kw = dict(quality=12, seed=6, rect=rect, wm_counter=wm)
        if search == "nonuniform":
            return fh.compress(img, metric=1, **kw), None
        if search == "statistics":
            out, st = fh.compress_with_stats(img, **kw)
            return out, st[:count]
        return fh.compress_with_selection(img, sels[first:first + count], **kw), None

    whole, stats = encode(None, 0, n)
    per_row = side // 4
    for rect, y0, rows in _row_rects(side, parts):
        first, count = y0 // 4 * per_row, rows // 4 * per_row
        out, st = encode(rect, first, count)
        a = whole.reshape(-1, 16)[first:first + count]
        b = out.reshape(-1, 16)[first:first + count]
        # each part starts its own watermark: solid blocks differ in it
        px = synth.blocks(img).reshape(n, 16)[first:first + count]
        searched = (px != px[:, :1]).any(axis=1)
        bad = np.nonzero((a != b).any(axis=1) & searched)[0]
        assert bad.size == 0, f"{bad.size} blocks differ from row {y0}, first {bad[:8]}"
        if stats is not None:
            assert stats[first:first + count].tobytes() == st.tobytes()


@pytest.mark.parametrize("threshold,side,parts", [(None, 640, 4), (0.6, 1280, 4), (1.5, 640, 4),
                                                  (1.5, 1280, 5)])
def test_parts_compose(fh, threshold, side, parts):
    """A large job equals its parts, which run the other form (the annealing
    streams are keyed by the block's place in the image).  threshold: of the
    learned search, None for the reference's.  At 1.5 every block falls back
    to the full search's candidates, a third of them rotations: the list of
    25600 blocks is then too long for one lane per pixel, and the rotations
    of 102400 too many for a phase of their own."""
    learned = threshold is not None
    img = synth.generate(side, side, 17)
    rk = None
    if learned:
        rk = fh.Ranker()
        rk.set_params(np.load(WEIGHTS))
    print(f"anneal forms threshold={threshold} {side}", flush=True)
    kw = dict(quality=50, seed=2, ranker=rk, threshold=threshold or 0.6)
    wm = ctypes.c_uint32(0xFFFFFFFF)
    whole = fh.compress(img, wm_counter=wm, **kw)
    wm2 = ctypes.c_uint32(0xFFFFFFFF)
    out = np.zeros_like(whole)
    for rect, _, _ in _row_rects(side, parts):
        fh.compress(img, wm_counter=wm2, rect=rect, out=out, **kw)
    bad = _diff(out, whole)
    assert bad.size == 0, f"{bad.size} blocks differ, first {bad[:8]}"
    assert wm.value == wm2.value
