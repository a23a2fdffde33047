"""GPU CSR transpose vs the CPU oracle, exact: tiles of 4,096 edges (one less,
one more, one only), one to four 8-bit passes over the columns, rows found from
the marks of their first entries (hub rows over many tiles, tiles among long
runs of empty rows, a tile of one-entry rows), duplicates, any column order."""
import numpy as np
import pytest
import torch

import oracle
from helpers import say

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ext():
    from dtc import load_extension
    return load_extension()


def sizes_of(kind, nnz, rng):
    if kind == "even":
        return np.bincount(rng.integers(0, max(1, nnz // 7), nnz), minlength=max(1, nnz // 7))
    if kind == "hub":  # one row holds most entries, empty rows on both sides
        s = np.zeros(700, np.int64)
        s[300] = nnz - nnz // 10
        s[rng.integers(301, 650, nnz // 10)] += 0
        s[640] = nnz // 10
        return s
    if kind == "sparse":  # far more rows than entries
        s = np.zeros(200000, np.int64)
        np.add.at(s, rng.integers(0, 200000, nnz), 1)
        return s
    return np.ones(nnz, np.int64)  # "ones"


@pytest.mark.parametrize("kind", ["even", "hub", "sparse", "ones"])
@pytest.mark.parametrize("K", [1, 256, 257, 65536, 65537, (1 << 24) + 1])
def test_transpose_shapes(ext, kind, K):
    rng = np.random.default_rng(K + len(kind))
    for nnz in (1, 4095, 4096, 4097, 30011):
        sizes = sizes_of(kind, nnz, rng)
        rowptr = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int32)
        col = rng.integers(0, K, nnz).astype(np.int32)
        col[-1] = K - 1
        M = sizes.shape[0]
        say("transpose", kind, f"M={M} K={K} nnz={nnz}")
        got = ext.csr_transpose(torch.from_numpy(rowptr).cuda(), torch.from_numpy(col).cuda(), M, K)
        for g, o in zip(got, oracle.csr_transpose(rowptr, col, M, K)):
            assert np.array_equal(g.cpu().numpy(), o)


@pytest.mark.parametrize("what", ["column", "negative", "order", "first", "last"])
def test_transpose_invalid(ext, what):
    rowptr = np.arange(0, 5001, 5).astype(np.int32)
    col = np.zeros(5000, np.int32)
    if what == "column":
        col[4999] = 10
    elif what == "negative":
        col[100] = -1
    elif what == "order":
        rowptr[500] = rowptr[501] + 1
    elif what == "first":
        rowptr[0] = 1
    else:
        rowptr[-1] = 4999
    with pytest.raises(RuntimeError, match="invalid CSR"):
        ext.csr_transpose(torch.from_numpy(rowptr).cuda(), torch.from_numpy(col).cuda(), 1000, 10)


def test_transpose_empty(ext):
    rpt, ct, perm = ext.csr_transpose(torch.zeros(4, dtype=torch.int32, device="cuda"),
                                      torch.empty(0, dtype=torch.int32, device="cuda"), 3, 5)
    assert rpt.tolist() == [0] * 6 and ct.numel() == 0 and perm.numel() == 0
