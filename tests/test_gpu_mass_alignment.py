"""fm_mass_p1_element_matrices into an array that starts at an odd double (8 bytes past a 16-byte boundary):
the same numbers as into an aligned one, and nothing outside it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("E", [1, 63, 64, 65, 1000])
def test_values_at_any_double(gpu, E):
    import torch

    from feelmri_amd import _lib, device

    r = np.random.default_rng(E)
    nodes = torch.tensor(r.normal(size=(50, 3)), device=gpu)
    elems = torch.tensor(np.stack([r.permutation(50)[:4] for _ in range(E)]).astype(np.int32), device=gpu)
    want = device.element_matrices(elems, nodes).reshape(-1)
    room = torch.full((16 * E + 2,), float("nan"), dtype=torch.float64, device=gpu)
    out = room[1:-1]
    assert out.data_ptr() % 16 == 8
    _lib.call("fm_mass_p1_element_matrices", E, device.ptr(elems), _lib.DTYPE_F64, device.ptr(nodes), device.ptr(out),
              device.stream_handle())
    assert torch.equal(out, want) and torch.isnan(room[0]) and torch.isnan(room[-1])
