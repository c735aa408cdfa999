"""The standalone block inverse over its sizes and layouts, against a float64
triangular solve."""
import numpy as np
import pytest
import scipy.linalg
import torch

from conftest import announce

pytestmark = pytest.mark.gpu


def _matrices(rng, mats, n):
    """Ancestor-masked A of random trees: strictly lower, entries around 0.2."""
    A = np.zeros((mats, n, n), np.float64)
    for m in range(mats):
        anc = np.zeros((n, n), bool)
        for i in range(1, n):
            p = int(rng.integers(0, i))
            anc[i] = anc[p]
            anc[i, p] = True
        A[m] = np.where(anc, rng.standard_normal((n, n)) * 0.3, 0)
    A += np.tril(rng.standard_normal((mats, n, n)) * (rng.random((mats, 1, 1)) < 0.5) * 0.1, -1)  # half of them dense
    return A.astype(np.float32)


# whole tiles (16-byte pieces), sizes on both sides of a tile, one row; offset:
# floats the buffer starts past a 16-byte boundary
@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 31, 32, 33, 47, 48, 63, 64])
@pytest.mark.parametrize("offset", [0, 1])
def test_block_inverse_sizes(cuda, n, offset):
    from dforktree_amd import ops
    announce(f"block inverse n={n} offset={offset}")
    rng = np.random.default_rng(n)
    mats = 37
    A = _matrices(rng, mats, n)
    junk = np.triu(np.full((n, n), 7.0, np.float32))  # the diagonal and above are not read
    buf = torch.full((mats * n * n + 8,), 5.0, device=cuda)
    x = buf[offset:offset + mats * n * n].view(mats, n, n)
    x.copy_(torch.from_numpy(A + junk))
    ops.block_inverse_(x)
    torch.cuda.synchronize()
    got = x.cpu().numpy().astype(np.float64)
    # forward substitution in fp32: each entry is a chain of at most n
    # multiply-adds, |error| <= n eps (|X| |A| |X|) entry by entry
    eps = 2.0 ** -24
    for m in range(mats):
        L = np.eye(n) + A[m].astype(np.float64)
        want = scipy.linalg.solve_triangular(L, np.eye(n), lower=True)
        bound = (n + 1) * eps * (np.abs(want) @ np.abs(L) @ np.abs(want)) + 1e-30
        assert np.all(np.abs(got[m] - want) <= bound)
        assert np.all(np.triu(got[m], 1) == 0) and np.all(np.diag(got[m]) == 1)
    assert torch.all(buf[:offset] == 5.0) and torch.all(buf[offset + mats * n * n:] == 5.0)  # nothing written around


def _forward_f32(A):
    """Forward substitution in fp32, row by row: what a non-finite value reaches."""
    n = A.shape[0]
    X = np.eye(n, dtype=np.float32)
    with np.errstate(all="ignore"):
        for i in range(n):
            for m in range(i):
                X[i] -= A[i, m] * X[m]
    return X


# a NaN in A, an infinity in A, and a row of X that overflows, in the middle
# and at the end of a 16-row block; whole tiles, an unaligned matrix, a size between
@pytest.mark.parametrize("n,offset,row", [(n, offset, row) for n, offset in ((16, 0), (32, 0), (64, 0), (64, 1), (40, 0))
                                          for row in (6, 15, 22, 31, 37, 63) if row < n])
def test_block_inverse_non_finite_rows(cuda, n, offset, row):
    from dforktree_amd import ops
    announce(f"block inverse non-finite n={n} offset={offset} row={row}")
    rng = np.random.default_rng(n + row)
    A = _matrices(rng, 1, n)[0]
    col = row // 2
    nan, inf, over = A.copy(), A.copy(), A.copy()
    nan[row, col] = np.nan
    inf[row, col] = np.inf
    over[row] = 0
    over[row - 1] = 0
    over[row, row - 1], over[row - 1, row - 2] = 1e30, 1e30  # X[row][row - 2] = +inf, the rest of the row 1e30 or 0 or 1
    over[row + 1:] = np.where(over[row + 1:] > 0, 0.5, 0)    # (no other row overflows by itself)
    bad = np.stack([nan, inf, over])
    buf = torch.zeros(2 * 3 * n * n + 8, device=cuda)
    x = buf[offset:offset + 2 * 3 * n * n].view(6, n, n)
    good = np.where(np.arange(n)[None, :, None] >= row, 0, bad)  # the same rows in front, zeros from `row` on
    x.copy_(torch.from_numpy(np.concatenate([bad, good]).astype(np.float32)))
    ops.block_inverse_(x)
    torch.cuda.synchronize()
    got = x.cpu().numpy()
    for c in range(3):
        # the rows in front do not see the row: the same bits as without it
        assert np.array_equal(got[c, :row].view(np.int32), got[3 + c, :row].view(np.int32)), c
        # from the row on: non-finite where the substitution's values are, and
        # nowhere else.  A non-finite element of A (0, 1) spreads over its row
        # as 0 * NaN; past its own 16 columns the sums here leave it out.
        want = _forward_f32(bad[c])
        upto = n if c == 2 else col + 1
        with np.errstate(all="ignore"):
            assert np.array_equal(np.isfinite(got[c, row:, :upto]), np.isfinite(want[row:, :upto])), c
            assert np.array_equal(np.isnan(got[c, row:, :upto]), np.isnan(want[row:, :upto])), c
            if c < 2 and (col // 16) * 16 + 16 < n:
                assert np.all(np.isfinite(got[c][:, (col // 16) * 16 + 16:])), c
    assert not np.isfinite(got[2, row, row - 2]) and got[2, row, row] == 1
