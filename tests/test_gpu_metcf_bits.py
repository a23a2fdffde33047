"""GPU ME-TCF build without sorts vs the CPU oracle, bit-exact.

Windows whose rows' columns strictly increase are numbered from column bitmaps
in LDS (kernels of 1 x 8, 4 x 8, 8 x 8, 8 x 16 and 16 x 16 waves x entries
per lane, taking spans of 2^20, then 2^21 columns; the 16 x 16 one at most
8,192 used 32-column pieces); larger windows from bitmaps of 2^16-column slices
and runs of 256 TC blocks.  Everything else is sorted.  Every output is an
integer or a copied value, so both sides are compared exactly."""
import numpy as np
import pytest

import oracle
from helpers import assert_metcf_equal, gpu_metcf, say

pytestmark = pytest.mark.gpu

CAPS = [64, 512, 2048, 4096, 8192, 16384]  # entries of the LDS kernels' largest window


@pytest.fixture(scope="module")
def ext():
    from dtc import load_extension
    return load_extension()


def csr(rows):
    rowptr = np.concatenate([[0], np.cumsum([len(r) for r in rows])]).astype(np.int32)
    return rowptr, np.concatenate([np.asarray(r) for r in rows]).astype(np.int32)


def check(ext, rows, ctx):
    rowptr, col = csr(rows)
    say("metcf", ctx, f"M={len(rows)} nnz={col.shape[0]}")
    values = np.random.default_rng(1).standard_normal(col.shape[0]).astype(np.float32)
    g = gpu_metcf(ext, rowptr, col, len(rows), 16, 8, values=values)
    o = oracle.metcf(rowptr, col, len(rows), 16, 8, values=values)
    assert_metcf_equal(g, o, ctx=ctx)
    assert np.array_equal(g["TCblockValues"], o["TCblockValues"]), ctx
    assert np.array_equal(np.sort(g["TCblockEdge"]), np.arange(col.shape[0])), ctx


def window(rng, entries, span, first=0):
    """16 rows of `entries` entries together, over exactly `span` columns."""
    span = max(span, -(-entries // 16))
    cuts = np.sort(rng.integers(0, entries + 1, 15))  # uneven rows, some empty
    sizes = np.diff(np.concatenate([[0], cuts, [entries]]))
    while sizes.max() > span:  # no row longer than the span
        i = int(sizes.argmax())
        over = sizes[i] - span
        sizes[i] = span
        sizes[int(sizes.argmin())] += over
    rows = [np.sort(rng.choice(span, n, replace=False)) for n in sizes]
    if entries >= 2 and span > 1:  # the span's first and last column
        i = int(sizes.argmax())
        if sizes[i] >= 2:
            rows[i][0], rows[i][-1] = 0, span - 1
    return [first + r for r in rows]


@pytest.mark.parametrize("blk_h", [24, 32])
@pytest.mark.parametrize("M", [1024 * 16, 1024 * 16 + 1])
def test_tall_windows(ext, M, blk_h):
    """Few windows of many rows: one workgroup plans the build up to 16,384 rows."""
    rng = np.random.default_rng(M + blk_h)
    rowptr, col = csr([np.sort(rng.choice(300, n, replace=False)) for n in rng.integers(0, 5, M)])
    say("metcf", "tall", M, blk_h)
    assert_metcf_equal(gpu_metcf(ext, rowptr, col, M, blk_h, 8), oracle.metcf(rowptr, col, M, blk_h, 8), ctx=(M, blk_h))


@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("cls", [1, 2, 3, 4, 5])
def test_spans_and_sizes(ext, monkeypatch, cls, wide):
    """Windows at the class's smallest and largest entry counts, spans at the
    edges of 32-column pieces, of their words and of the kernel's limit, and a
    first column other than 0; with wider windows among them, which the first
    rows (of one entry) do not show."""
    monkeypatch.setenv("DTC_METCF_PATH", "auto")
    rng = np.random.default_rng(70 + cls)
    lo, cap = CAPS[cls - 1], CAPS[cls]
    limit = 1 << (20 if cls == 1 else 21)
    rows = []
    for E in (lo + 1, lo + 63, cap - 1, cap):
        for span in (E // 16, 31 + E // 16, 1023, 1024, 1025, 4097, limit - 1, limit):
            rows += window(rng, E, span, first=int(rng.integers(0, 5)) * 777)
        for span in (limit + 1, 3 * limit) if wide else ():
            w = window(rng, E - 1, span)
            w[0], w[1] = [5], np.union1d(w[0], w[1])
            rows += w
    rows += [[], [3]]  # a last window of two rows
    check(ext, rows, f"class {cls} spans")


@pytest.mark.parametrize("kind", ["swap", "duplicate", "descending row", "pieces"])
def test_left_to_the_sort(ext, monkeypatch, kind):
    """Windows that the bit kernels must leave, among windows that they take:
    one pair out of order, one duplicate, in each class (first rows sorted),
    one row descending, more 32-column pieces than the largest kernel keeps."""
    monkeypatch.setenv("DTC_METCF_PATH", "auto")
    rng = np.random.default_rng(90 + len(kind))
    rows = []
    for cap in CAPS[1:]:
        for bad in (False, True):
            w = window(rng, cap - 3, 1 << 18)
            if kind == "pieces":
                w = [np.sort(rng.choice(1 << 16, cap // 16, replace=False)) * 32 for _ in range(16)]
            elif bad:
                i = 15 - int(np.argmax([len(r) >= 3 for r in w[::-1]]))
                if kind == "swap":
                    w[i][[-2, -1]] = w[i][[-1, -2]]
                elif kind == "duplicate":
                    w[i][1] = w[i][0]
                else:
                    w[i] = w[i][::-1].copy()
            rows += w
    check(ext, rows, kind)


@pytest.mark.parametrize("kind", ["duplicate", "swap"])
@pytest.mark.parametrize("first", [0, 1, 1000])
@pytest.mark.parametrize("cls", [1, 2, 3, 4, 5])
def test_defect_between_slots(ext, monkeypatch, cls, first, kind):
    """Windows whose only duplicate, or only descent, lies between local entries
    64 j - 1 and 64 j of one row, the two held by different slots of a lane or
    by different waves, with a first column of 0 and above; among sorted ones."""
    monkeypatch.setenv("DTC_METCF_PATH", "auto")
    rng = np.random.default_rng(500 + cls)
    cap = CAPS[cls]
    per_wave = 64 * (16 if cls >= 4 else 8)  # entries of a wave
    rows = []
    # a wave's first and last boundary, the window's last, and (larger classes) waves' ends
    for at in sorted({64, per_wave - 64, cap - 64} | ({per_wave, cap - per_wave} if cap > per_wave else set())):
        # short rows around one that holds entries at - 40 .. at + 39
        sizes = [(at - 40) // 8] * 7 + [(at - 40) // 8 + (at - 40) % 8] + [80] + [(cap - at - 40) // 7] * 7
        w = [first + np.sort(rng.choice(1 << 14, n, replace=False)) for n in sizes]
        if kind == "duplicate":
            w[8][40] = w[8][39]
        else:
            w[8][[39, 40]] = w[8][[40, 39]]
        rows += w + window(rng, cap - 3, 1 << 14, first=first)
    check(ext, rows, f"class {cls} {kind} between slots, first {first}")


@pytest.mark.parametrize("span", [16384, (1 << 16) - 1, 1 << 16, (1 << 16) + 1, 300000])
def test_large_windows(ext, monkeypatch, span):
    """Windows beyond the LDS kernels: spans at the edges of a slice, full rows
    (runs of 32,768 entries), an empty slice, and a last window of 5 rows."""
    monkeypatch.setenv("DTC_METCF_PATH", "auto")
    rng = np.random.default_rng(span)
    rows = window(rng, 16385, span) + window(rng, 60001, span)
    rows += [np.arange(3000) for _ in range(16)]  # 375 full TC blocks
    rows += [np.concatenate([np.arange(1000), span - 1000 + np.arange(1000)]) for _ in range(16)]
    rows += window(rng, 40, span)
    rows += [np.sort(rng.choice(span, 9000, replace=False)) for _ in range(5)]
    check(ext, rows, f"large windows over {span}")


@pytest.mark.parametrize("at", ["first", "middle", "last"])
def test_large_windows_unsorted(ext, monkeypatch, at):
    """One pair out of order in one row of one large window: all of them go
    through the sort."""
    monkeypatch.setenv("DTC_METCF_PATH", "auto")
    rng = np.random.default_rng(5)
    rows = [np.sort(rng.choice(1 << 17, 1500, replace=False)) for _ in range(48)]
    r = {"first": rows[0], "middle": rows[23], "last": rows[47]}[at]
    r[[-2, -1]] = r[[-1, -2]]
    check(ext, rows, f"large unsorted {at}")


@pytest.mark.parametrize("width", [1, 8, 200])
def test_every_window_global(ext, monkeypatch, width):
    """Every window through the large windows' kernels (when the bitmaps fit
    the workspace) or their sort: windows of few entries, many empty ones."""
    monkeypatch.setenv("DTC_METCF_PATH", "global")
    rng = np.random.default_rng(width)
    rows = []
    for _ in range(40):
        rows += window(rng, 16 * width, 5000) if rng.random() < 0.7 else [[]] * 16
    check(ext, rows, f"global width {width}")


def test_negative_column_inside_a_row(ext, monkeypatch):
    """A negative column that is not its row's first is still refused."""
    monkeypatch.setenv("DTC_METCF_PATH", "auto")
    rows = [np.arange(20) + i for i in range(16)]
    rows[7][-1] = -5
    rowptr, col = csr(rows)
    with pytest.raises(RuntimeError, match="negative column"):
        gpu_metcf(ext, rowptr, col, 16, 16, 8)


@pytest.mark.parametrize("windows", [1, 64, 1023, 1024, 1025, 4095, 4096, 4097])
def test_window_counts(ext, monkeypatch, windows):
    """Builds at the edges of the one-workgroup plan (1,024 windows) and of the
    one-workgroup offsets (4,096), with empty windows, a last window of one row,
    one window of each LDS class and one beyond them."""
    monkeypatch.setenv("DTC_METCF_PATH", "auto")
    rng = np.random.default_rng(windows)
    M = windows * 16 - 15
    rows = [np.sort(rng.choice(60000, n, replace=False)) for n in rng.integers(0, 3, M)]
    for i in range(min(windows, 200)):  # empty windows
        w = int(rng.integers(0, windows))
        rows[w * 16:w * 16 + 16] = [[] for _ in rows[w * 16:w * 16 + 16]]
    for n in (300, 1500, 3000, 7000, 15000, 40000):
        rows[int(rng.integers(0, M))] = np.sort(rng.choice(60000, n, replace=False))
    check(ext, rows, f"{windows} windows")


@pytest.mark.parametrize("windows", [40, 2000])
def test_row_pointer_beyond_the_edges(ext, windows):
    """A row pointer that would put a window's entries far outside the edge
    arrays is refused before anything reads them."""
    rowptr = np.arange(windows * 16 + 1, dtype=np.int32)
    rowptr[100] = 2_000_000_000
    with pytest.raises(RuntimeError, match="nodePointer decreases"):
        gpu_metcf(ext, rowptr, np.zeros(windows * 16, np.int32), windows * 16, 16, 8)


@pytest.mark.parametrize("repeat", [False, True])
@pytest.mark.parametrize("every", [1, 7, 400])
def test_unsorted_rows_among_many(ext, monkeypatch, every, repeat):
    """A repeated entry or a descent in one row of every window, of some and of
    one or two, in any of the 16 rows: found by the look at each window or by its
    own kernel."""
    monkeypatch.setenv("DTC_METCF_PATH", "auto")
    rng = np.random.default_rng(every + repeat)
    rows = []
    for w in range(700):
        rows += window(rng, int(rng.choice([90, 300, 700, 2500])) if w % 50 else 5000, 9000, first=w % 3)
        if w % every == every // 2:
            r = max(range(len(rows) - 16, len(rows)), key=lambda i: (len(rows[i]) >= 3) * rng.random())
            if len(rows[r]) >= 2:
                i = int(rng.integers(0, len(rows[r]) - 1))
                rows[r][i:i + 2] = rows[r][i:i + 1] if repeat else rows[r][i:i + 2][::-1].copy()
    check(ext, rows, ("unsorted rows", every, repeat))
