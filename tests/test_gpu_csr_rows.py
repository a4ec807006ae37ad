"""CSR product with two rows a lane group (one or two encodings, long calls): the rows of a pair are of
any length, and a row's sum has the same bits as in a short call, where a group has one row."""
import numpy as np
import pytest
import scipy.sparse as sp
import torch

pytestmark = pytest.mark.gpu

N = 16 * 32 * 256  # rows from which 256 CUs have two rounds of pairs


@pytest.mark.parametrize("V", [1, 2])
@pytest.mark.parametrize("n_rows", [N - 32, N - 31, N, N + 1, N + 17])
def test_pairs_of_rows_of_any_length(gpu, n_rows, V):
    from feelmri_amd import device

    rng = np.random.default_rng(n_rows)
    lengths = rng.choice([0, 1, 14, 15, 16, 17, 33], size=n_rows)
    lengths[-1] = 40
    indptr = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int64)
    indices = rng.integers(0, n_rows, size=indptr[-1]).astype(np.int64)
    data = rng.standard_normal(indptr[-1])
    x = rng.standard_normal((n_rows, V)) + 1j * rng.standard_normal((n_rows, V))
    to = lambda a: torch.from_numpy(a).to(gpu)
    p, i, d, xd = to(indptr), to(indices), to(data), to(x)

    got = device.csr_spmv(p, i, d, xd).cpu().numpy()
    short = 1000  # the last rows as a call of their own
    tail = device.csr_spmv(p[-short - 1:].contiguous(), i, d, xd).cpu().numpy()
    np.testing.assert_array_equal(got[-short:].view(np.float64), tail.view(np.float64))

    # n terms of one sign or another: n roundings of the sum of their sizes, in each part and
    # on each side
    M = sp.csr_matrix((data, indices, indptr), shape=(n_rows, n_rows))
    bound = 2 * np.sqrt(2) * lengths[:, None] * 2.0**-53 * (abs(M) @ np.abs(x))
    assert np.all(np.abs(got - M @ x) <= bound)
