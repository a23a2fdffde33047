"""SDDMM over the widths and row shapes at which its kernels change form,
against the float64 dot products."""
import numpy as np
import pytest
import torch

from helpers import say

pytestmark = pytest.mark.gpu

# rows of every length and gaps between them: rows far longer than a wave's 64
# edges, rows of one entry each, empty rows, and both mixed
SHAPES = {
    "long": [700, 3, 0, 200, 65, 64, 63],
    "single": [1, 0, 0] * 150,
    "mixed": ([1] * 40 + [0] * 30 + [90] + [7] * 25) * 3,
    "short": [9] * 133,
    "one": [1],
}


def run(shape, n, dtype, give_rows, y_rows=800):
    from dtc import load_extension
    ext = load_extension()
    lengths = np.array(SHAPES[shape])
    rng = np.random.default_rng(n + len(lengths))
    M, K = len(lengths), 800
    rowptr = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int32)
    col = np.concatenate([np.sort(rng.choice(K, k, replace=False)) for k in lengths]).astype(np.int32)
    row = np.repeat(np.arange(M), lengths)
    X = torch.from_numpy(rng.standard_normal((M, n)).astype(np.float32)).cuda()
    Y = torch.from_numpy(rng.standard_normal((y_rows, n)).astype(np.float32)).to(dtype).cuda()
    bad = sorted(set(range(y_rows)) - set(col.tolist()))
    if bad:  # a row of Y that no edge names
        Y[bad[0]] = float("inf")
    rows = torch.from_numpy(row.astype(np.int32)).cuda() if give_rows else None
    say("sddmm", shape, n, dtype, give_rows, y_rows)
    out = ext.sddmm_csr(torch.from_numpy(rowptr).cuda(), torch.from_numpy(col).cuda(), X, Y, rows).cpu().numpy()
    inside = col < y_rows
    a, b = X.double().cpu().numpy()[row], Y.double().cpu().numpy()[np.minimum(col, y_rows - 1)]
    a[~inside] = b[~inside] = 0.0  # columns past Y give 0
    # a float32 sum of n products: (n + 4) 2^-24 of the sum of magnitudes
    assert np.all(np.abs(out - (a * b).sum(1)) <= (n + 4) * 2.0 ** -24 * np.abs(a * b).sum(1)), (shape, n)


@pytest.mark.parametrize("shape", sorted(SHAPES))
@pytest.mark.parametrize("n", [1, 3, 4, 5, 31, 60, 63, 64, 65, 100, 127, 128, 130, 191, 192, 193, 196, 256, 300])
def test_float32(shape, n):
    run(shape, n, torch.float32, True)


@pytest.mark.parametrize("shape", sorted(SHAPES))
@pytest.mark.parametrize("n", [4, 8, 20, 64, 72, 120, 128, 136, 200, 256, 264])
def test_bfloat16(shape, n):
    run(shape, n, torch.bfloat16, True)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n", [16, 128])
def test_rows_searched_and_short_y(n, dtype):
    run("mixed", n, dtype, False)
    run("mixed", n, dtype, True, y_rows=500)


@pytest.mark.parametrize("shape", ["mixed", "single"])
@pytest.mark.parametrize("n,dtype", [(4, torch.float32), (64, torch.float32), (65, torch.float32),
                                     (128, torch.float32), (192, torch.float32), (193, torch.float32),
                                     (8, torch.bfloat16), (128, torch.bfloat16), (256, torch.bfloat16),
                                     (264, torch.bfloat16)])
def test_columns_past_y_of_nonfinite_rows(shape, n, dtype):
    """An edge whose column Y does not have gives 0 at every width, also where
    its row of X holds infinities or NaN."""
    from dtc import load_extension
    ext = load_extension()
    lengths = np.array(SHAPES[shape])
    rng = np.random.default_rng(n)
    M, y_rows = len(lengths), 300
    rowptr = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int32)
    col = np.concatenate([np.sort(rng.choice(800, k, replace=False)) for k in lengths]).astype(np.int32)
    row = np.repeat(np.arange(M), lengths).astype(np.int32)
    Xn = rng.standard_normal((M, n)).astype(np.float32)
    # rows whose edges are all past Y become non-finite
    past = np.array([len(c) > 0 and (c >= y_rows).all() for c in np.split(col, rowptr[1:-1])])
    Xn[past] = np.inf
    Xn[np.flatnonzero(past)[::2], 0] = np.nan
    X = torch.from_numpy(Xn).cuda()
    Y = torch.from_numpy(rng.standard_normal((y_rows, n)).astype(np.float32)).to(dtype).cuda()
    say("sddmm short y, non-finite x", shape, n, dtype, int(past.sum()))
    assert past.any()
    out = ext.sddmm_csr(torch.from_numpy(rowptr).cuda(), torch.from_numpy(col).cuda(), X, Y,
                        torch.from_numpy(row).cuda()).cpu().numpy()
    inside = col < y_rows
    assert np.array_equal(out[~inside], np.zeros((~inside).sum(), np.float32))
    a, b = Xn.astype(np.float64)[row], Y.double().cpu().numpy()[np.minimum(col, y_rows - 1)]
    a[~inside] = b[~inside] = 0.0
    assert np.all(np.abs(out - (a * b).sum(1)) <= (n + 4) * 2.0 ** -24 * np.abs(a * b).sum(1))
