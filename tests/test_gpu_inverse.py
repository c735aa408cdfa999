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
# floats the buffer starts past a 16-byte boundary (row-by-row form)
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
