"""Node splits of the t-grouped direct sum: meshes around the split sizes (256 and 2048 nodes), with the
workspace the query reports, with less (fewer splits) and with too little, and the tile that asks for
the most LDS (32 groups, 4 encodings, 32 modes, FP64).  Against the FP64 oracle; tolerances as in the tests of
the groups: mixed 1e-5, FP64 1e-10."""
import ctypes

import numpy as np
import pytest
import scipy.sparse as sp

from test_gpu_groups import TOL, _samples
from test_gpu_signal import _nodes, rel_l2

pytestmark = pytest.mark.gpu


def _execute(plan, nodes, precision, motion, ws_bytes):
    """fm_signal_execute with a workspace of ws_bytes; (status, samples)."""
    import torch

    from feelmri_amd import _lib, device

    modes, coef = motion if motion is not None else (None, None)
    out = torch.full((plan.n_samples, nodes.n_enc), float("nan"), dtype=torch.complex128, device=plan.device)
    ws = torch.empty(max(1, ws_bytes), dtype=torch.uint8, device=plan.device)
    rc = _lib.load().fm_signal_execute(
        plan._h, device._prec(precision), ctypes.c_int64(nodes.n_nodes), nodes.n_enc, device.ptr(nodes.packed),
        device.ptr(modes), 0 if modes is None else modes.shape[0] // 3, device.ptr(coef), device.ptr(ws),
        ctypes.c_size_t(ws_bytes), device.ptr(out), device.stream_handle())
    return rc, out.cpu().numpy()


@pytest.mark.parametrize("n", [1, 255, 257, 2048, 2049, 5000])
@pytest.mark.parametrize("precision", ["mixed", "f64"])
@pytest.mark.parametrize("moving", [False, True])
def test_splits_and_workspaces(gpu, n, precision, moving):
    import torch

    import oracle
    from feelmri_amd import _lib, device

    V, R = 2, 3
    kloc, t = _samples([17, 20, 33, 16, 31, 40], False, False)
    rng = np.random.default_rng(n)
    r0, phi, T2, mxy, _ = _nodes(n, V, 5)
    plan = device.SignalPlan(kloc, t, method="direct")
    nodes = device.SignalNodes.from_arrays(r0, phi, T2, mxy)
    motion, pod = None, None
    if moving:
        modes = rng.normal(0, 1e-3, (3 * R, n)).astype(np.float32)
        coef = np.concatenate([rng.normal(size=(plan.n_tgroups, R)), np.zeros((plan.n_tgroups, 3))], axis=1)
        motion = (torch.tensor(modes, device=gpu), torch.tensor(coef, device=gpu))
        m3 = modes.astype(float).reshape(3, R, n)
        at = {float(tt): np.einsum("crn,r->nc", m3, c[:R]) for tt, c in zip(plan.tgroup_t, coef)}
        pod = lambda tt: at[float(tt)]  # noqa: E731
    want = oracle.Signal(0, sp.identity(n, format="csr"), kloc, t, r0, phi, T2, mxy, pod)
    want = np.asarray(want).reshape(-1, V)
    full = plan.workspace_bytes(precision, n, V, moving=moving)
    one = plan.n_samples * V * 16
    least = one * -(-n // 2048) if n > 2048 else 0
    for ws in sorted({full, (full + least) // 2, least, 64 << 20}):
        rc, got = _execute(plan, nodes, precision, motion, ws)
        assert rc == _lib.FM_OK, (ws, full)
        assert rel_l2(got, want) <= TOL[precision], (ws, full)
    if least:
        assert _execute(plan, nodes, precision, motion, least - 16)[0] == _lib.FM_ERR_WORKSPACE


@pytest.mark.parametrize("R", [31, 32])
def test_largest_lds_tile(gpu, R):
    """Groups of 8 or 9 samples: 32 groups to a tile, with 4 of 5 encodings a launch."""
    import torch

    import oracle
    from feelmri_amd import device

    n, V = 300, 5
    kloc, t = _samples([8, 9] * 40, False, False)
    rng = np.random.default_rng(R)
    r0, phi, T2, mxy, _ = _nodes(n, V, 5)
    plan = device.SignalPlan(kloc, t, method="direct")
    nodes = device.SignalNodes.from_arrays(r0, phi, T2, mxy)
    modes = rng.normal(0, 1e-3, (3 * R, n)).astype(np.float32)
    coef = np.concatenate([rng.normal(size=(plan.n_tgroups, R)), np.zeros((plan.n_tgroups, 3))], axis=1)
    m3 = modes.astype(float).reshape(3, R, n)
    at = {float(tt): np.einsum("crn,r->nc", m3, c[:R]) for tt, c in zip(plan.tgroup_t, coef)}
    want = np.asarray(oracle.Signal(0, sp.identity(n, format="csr"), kloc, t, r0, phi, T2, mxy, lambda tt: at[float(tt)]))
    for precision in ("f64", "mixed"):
        got = plan.execute(nodes, precision=precision, motion=(torch.tensor(modes, device=gpu),
                                                              torch.tensor(coef, device=gpu))).cpu().numpy()
        assert rel_l2(got, want.reshape(-1, V)) <= TOL[precision]
