"""Sizes where the mass kernels' tiles end: element matrices around a
wavefront's and a workgroup's elements (both node types), CSR products around
a group of rows' and a workgroup's rows, empty rows and rows longer than a
group's 16 lanes, encodings around the 4 taken together.

Tolerances: both are FP64 sums of at most a few dozen like terms, 1e-13.
"""
import numpy as np
import pytest
import scipy.sparse as sp

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("E", [1, 7, 8, 63, 64, 65, 255, 257, 2049])
def test_element_matrices_sizes(gpu, E, dtype):
    import torch

    from feelmri_amd import device

    rng = np.random.default_rng(E)
    nodes = rng.normal(size=(50, 3)).astype(dtype)
    elems = np.array([rng.choice(50, 4, replace=False) for _ in range(E)], dtype=np.int32)
    X = nodes[elems].astype(np.float64)
    vol = np.abs(np.linalg.det(X[:, 1:] - X[:, :1])) / 6
    want = vol[:, None, None] / 20 * (1 + np.eye(4))
    got = device.element_matrices(torch.from_numpy(elems).to(gpu), torch.from_numpy(nodes).to(gpu)).cpu().numpy()
    assert np.abs(got.reshape(E, 4, 4) - want).max() <= 1e-13 * np.abs(want).max()


@pytest.mark.parametrize("V", [1, 2, 3, 4, 5, 9])
@pytest.mark.parametrize("n_rows", [1, 15, 16, 63, 65, 129, 1030])
def test_csr_product_sizes(gpu, n_rows, V):
    import torch

    from feelmri_amd import device

    rng = np.random.default_rng(10 * n_rows + V)
    n_cols = 97
    lens = rng.choice([0, 1, 15, 16, 17, 50], n_rows)
    lens[-1] = 17
    A = sp.csr_matrix((rng.normal(size=lens.sum()),
                       np.concatenate([rng.choice(n_cols, k, replace=False) for k in lens]),
                       np.concatenate([[0], np.cumsum(lens)])), shape=(n_rows, n_cols))
    x = rng.normal(size=(n_cols, V)) + 1j * rng.normal(size=(n_cols, V))
    got = device.csr_spmv(torch.from_numpy(A.indptr.astype(np.int64)).to(gpu),
                          torch.from_numpy(A.indices.astype(np.int64)).to(gpu),
                          torch.from_numpy(A.data).to(gpu), torch.from_numpy(x).to(gpu)).cpu().numpy()
    want = A @ x
    assert got.shape == want.shape and np.abs(got - want).max() <= 1e-13 * np.abs(x).max() * np.sqrt(50)
