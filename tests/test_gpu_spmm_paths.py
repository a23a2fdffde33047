"""The SpMM kernels' forms at the sizes where they change: ragged widths, one
to several element loads per group, windows split over a workgroup, several
windows per wave; each against the float64 CSR product."""
import numpy as np
import pytest
import torch

import oracle
from helpers import say

pytestmark = pytest.mark.gpu


def random_csr(rng, rows, cols, lengths):
    """Rows of the given lengths with distinct sorted columns."""
    rowptr = np.zeros(rows + 1, np.int64)
    rowptr[1:] = np.cumsum(lengths)
    col = np.concatenate([np.sort(rng.choice(cols, k, replace=False)) for k in lengths] or [np.zeros(0, np.int64)])
    values = rng.uniform(-1, 1, col.shape[0]).astype(np.float32)
    return rowptr.astype(np.int32), col.astype(np.int32), values


def check(rowptr, col, values, cols, n, schedule, **options):
    """Componentwise: a float32 sum of k products is off by at most
    (k + 4) 2^-24 of the sum of their magnitudes."""
    from dtc.matrix import DTCMatrix
    rows = rowptr.shape[0] - 1
    A = DTCMatrix(rowptr, col, values, num_rows=rows, num_cols=cols)
    B = np.random.default_rng(n).standard_normal((cols, n)).astype(np.float32)
    out = torch.full((rows, n), float("nan"), device="cuda")
    say("spmm path", rows, cols, n, schedule, options)
    C = A.spmm(torch.from_numpy(B).cuda(), schedule=schedule, out=out, **options).cpu().numpy()
    exact, mag = oracle.spmm_csr_f64(rowptr, col, values, B, rows, with_abs=True)
    bound = (np.diff(rowptr)[:, None] + 4) * 2.0 ** -24 * mag
    assert np.all(np.abs(C - exact) <= bound), (n, schedule, options)


@pytest.mark.parametrize("schedule", ["windows", "balanced"])
@pytest.mark.parametrize("n", [1, 3, 5, 15, 17, 31, 33, 47, 63, 65, 72, 97, 130, 191, 260])
def test_ragged_widths(n, schedule):
    """Widths that no vector divides: the last lanes of a row move back."""
    rng = np.random.default_rng(n)
    lengths = rng.integers(0, 20, 330)
    lengths[160:200] = 0  # two empty windows
    check(*random_csr(rng, 330, 200, lengths), 200, n, schedule)


@pytest.mark.parametrize("schedule,options", [("windows", {}), ("balanced", {}), ("balanced", {"chunk_blocks": 5}),
                                              ("balanced", {"deterministic": True, "chunk_blocks": 4})])
@pytest.mark.parametrize("fill", [0.05, 0.2, 0.45, 0.7, 1.0])
def test_elements_per_group(fill, schedule, options):
    """Groups from a few elements to all 512: the first load's 64 (or 256),
    the second's, and the loop past them."""
    rng = np.random.default_rng(int(fill * 100))
    lengths = np.full(150, int(fill * 96))
    lengths[40:60] = 3  # a sparse window among them
    check(*random_csr(rng, 150, 96, lengths), 96, 64, schedule, **options)


@pytest.mark.parametrize("n", [16, 64, 100])
@pytest.mark.parametrize("rows,long_row", [(16, 500), (15, 33), (1000, 900), (3000, 0)])
def test_split_windows(rows, long_row, n):
    """Few windows: each is shared by four waves, from none to many groups."""
    rng = np.random.default_rng(rows)
    lengths = rng.integers(4, 12, rows)
    if rows > 100:
        lengths[64:80] = 0
        lengths[80:96] = 0
        lengths[80] = 1  # a window of one entry
    lengths[rows // 2] = max(long_row, lengths[rows // 2])
    check(*random_csr(rng, rows, 1200, lengths), 1200, n, "windows")


def test_several_windows_per_wave():
    """Many short windows, empty ones among them, a ragged last one."""
    rng = np.random.default_rng(9)
    rows = 16 * 17000 + 5
    lengths = rng.integers(0, 3, rows)
    lengths[1600:4800] = 0
    lengths[-21:] = 2
    check(*random_csr(rng, rows, 500, lengths), 500, 260, "windows")


@pytest.mark.parametrize("n", [16, 33, 64, 96, 320])
@pytest.mark.parametrize("windows", [2301, 40000])
def test_long_windows(n, windows):
    """Hub windows among short ones (several short ones per wave at 40,000
    windows): below, at and above the 128 blocks from which a workgroup shares
    a window, neighbours, the first and the last window."""
    rng = np.random.default_rng(windows + n)
    cols = 3000 if windows < 10000 else 1300
    rows = windows * 16 - 3
    lengths = rng.integers(0, 2, rows)
    lengths[16 * 8:16 * 10] = 0
    for w, blocks in ((0, 160), (5, 127), (20, 128), (21, 129), (22, 130), (40, 132), (41, 160), (windows - 1, 159)):
        lengths[16 * w:16 * (w + 1)] = 0
        lengths[min(16 * w + 7, rows - 1)] = 8 * blocks - 3
    check(*random_csr(rng, rows, cols, lengths), cols, n, "windows")


@pytest.mark.parametrize("n,options", [(128, {}), (130, {}), (64, {"vec": 1}), (192, {"vec": 2})])
@pytest.mark.parametrize("rows", [16 * 2301 - 3, 16 * 2304])
def test_long_windows_wide_b(rows, n, options):
    """B beyond 256 MB: the column tiles go one after another, the hub windows of
    all tiles before the others; group counts that are and are not a multiple of
    8 and of 4, hub windows in every quarter, next to each other and at both
    ends."""
    rng = np.random.default_rng(rows + n)
    cols = (1 << 28) // (4 * n) + 1000
    windows = -(-rows // 16)
    lengths = rng.integers(0, 3, rows)
    lengths[16 * 800:16 * 808] = 0
    for w in (0, 1, 2, 3, 4, 575, 576, 1150, 1151, 1152, 1727, windows - 2, windows - 1):
        lengths[min(16 * w + 7, rows - 1)] = 8 * 129 + w % 64
    # rows with a hub's length pick from all of B's rows: distinct by construction
    rowptr = np.zeros(rows + 1, np.int64)
    rowptr[1:] = np.cumsum(lengths)
    col = np.concatenate([np.sort((rng.integers(0, cols) + np.arange(k) * (cols // 1200)) % cols) for k in lengths])
    values = rng.uniform(-1, 1, col.shape[0]).astype(np.float32)
    check(rowptr.astype(np.int32), col.astype(np.int32), values, cols, n, "windows", **options)


@pytest.mark.parametrize("n,options", [(130, {}), (256, {}), (64, {"vec": 1, "deterministic": True}), (160, {"vec": 2}),
                                       (130, {"chunk_blocks": 8, "cut_span_blocks": 64})])
def test_balanced_wide_b(n, options):
    """B beyond 256 MB in three, four and five column tiles, two of them at a
    time; with a cut span side by side."""
    rng = np.random.default_rng(n)
    cols = (1 << 28) // (4 * n) + 1000
    rows = 16 * 90 - 5
    lengths = rng.integers(0, 20, rows)
    lengths[160:192] = 0
    lengths[400] = 1100
    rowptr = np.zeros(rows + 1, np.int64)
    rowptr[1:] = np.cumsum(lengths)
    col = np.concatenate([np.sort((rng.integers(0, cols) + np.arange(k) * (cols // 1200)) % cols) for k in lengths])
    values = rng.uniform(-1, 1, col.shape[0]).astype(np.float32)
    check(rowptr.astype(np.int32), col.astype(np.int32), values, cols, n, "balanced", **options)


@pytest.mark.parametrize("n", [48, 64, 65, 96, 97, 224])
@pytest.mark.parametrize("blocks", [8800, 8801, 17600, 17601, 35200, 35201])
def test_default_chunks(n, blocks):
    """Balanced runs with the default chunk and lane shape, at block counts
    where the chunk doubles from 8 to 16 for four, two and one 64 columns."""
    rng = np.random.default_rng(blocks + n)
    rows = 16 * (blocks // 4)
    lengths = np.zeros(rows, np.int64)
    lengths[::16] = 25  # four blocks a window
    lengths[16 * 3] = 24 + 8 * (blocks % 4) + 1
    check(*random_csr(rng, rows, 400, lengths), 400, n, "balanced")


@pytest.mark.parametrize("n", [64, 65, 192, 193])
@pytest.mark.parametrize("blocks", [31, 32, 33])
def test_even_windows(n, blocks):
    """Balanced runs with the default chunk over windows of one length, a little
    below, at and above a power of two, where the chunk keeps windows whole."""
    rng = np.random.default_rng(blocks + n)
    rows = 16 * 301 - 3
    lengths = np.zeros(rows, np.int64)
    lengths[::16] = 8 * blocks - 2
    check(*random_csr(rng, rows, 700, lengths), 700, n, "balanced")


@pytest.mark.parametrize("deterministic", [False, True])
def test_balanced_workspace_by_block_count(deterministic):
    """A workspace sized by the chunk of the block count alone, or for a wider N:
    accepted for a narrow N, whose default chunks are shorter."""
    from dtc.capi import Library
    from dtc.matrix import DTCMatrix
    lib = Library()
    rng = np.random.default_rng(9)
    rows, n = 16 * 3000, 64
    lengths = np.zeros(rows, np.int64)
    lengths[::16] = 32
    rowptr, col, values = random_csr(rng, rows, 400, lengths)
    A = DTCMatrix(rowptr, col, values, num_rows=rows, num_cols=400)
    B = rng.standard_normal((400, n)).astype(np.float32)
    Bd = torch.from_numpy(B).cuda()
    exact, mag = oracle.spmm_csr_f64(rowptr, col, values, B, rows, with_abs=True)
    opt = lib.options(deterministic=deterministic)
    chunks = -(-A.block_count // 32)
    formula = 256 + 8 * chunks
    if deterministic:
        formula = -(-formula // 256) * 256 + 2 * chunks * 16 * 128 * 4
    for bytes_ in (formula, lib.spmm_balanced_workspace_size(A.block_count, 4096, opt)):
        C = torch.full((rows, n), float("nan"), device="cuda")
        ws = torch.empty(bytes_, dtype=torch.uint8, device="cuda")
        say("balanced workspace", bytes_)
        lib.spmm_balanced(A.tcblock_rowid.data_ptr(), A.tcblocktile_id.data_ptr(), A.tcblock_offset.data_ptr(),
                          A.sparse_atox.data_ptr(), A.values_tc.data_ptr(), A.block_count, A.nnz, rows, Bd.data_ptr(),
                          400, n, C.data_ptr(), ws.data_ptr(), bytes_, options=opt,
                          stream=torch.cuda.current_stream().cuda_stream)
        assert np.all(np.abs(C.cpu().numpy() - exact) <= 36 * 2.0 ** -24 * mag)


def test_noalloc_default_chunk():
    """The allocation-free entry point with the default chunk: the ordered merge
    of 12,000 blocks at N = 128 exceeds its scratch in chunks of 8 and fits it in
    chunks of 32."""
    from dtc.capi import Library
    from dtc.matrix import DTCMatrix
    lib = Library()
    rng = np.random.default_rng(8)
    rows, n = 16 * 3000, 128
    lengths = np.zeros(rows, np.int64)
    lengths[::16] = 32
    rowptr, col, values = random_csr(rng, rows, 400, lengths)
    A = DTCMatrix(rowptr, col, values, num_rows=rows, num_cols=400)
    B = rng.standard_normal((400, n)).astype(np.float32)
    C = torch.full((rows, n), float("nan"), device="cuda")
    Bd = torch.from_numpy(B).cuda()
    opt = lib.options(deterministic=True)
    say("noalloc default chunk", A.block_count)
    lib.spmm_balanced_noalloc(A.tcblock_rowid.data_ptr(), A.tcblocktile_id.data_ptr(), A.tcblock_offset.data_ptr(),
                              A.sparse_atox.data_ptr(), A.values_tc.data_ptr(), A.block_count, A.nnz, rows,
                              Bd.data_ptr(), 400, n, C.data_ptr(), options=opt,
                              stream=torch.cuda.current_stream().cuda_stream)
    exact, mag = oracle.spmm_csr_f64(rowptr, col, values, B, rows, with_abs=True)
    assert np.all(np.abs(C.cpu().numpy() - exact) <= 36 * 2.0 ** -24 * mag)
