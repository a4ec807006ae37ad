"""The direct sum over samples grouped by t against the FP64 oracle, at the
sizes where its tiling can go wrong: groups of 1 to 600 samples (a lane takes
two samples of a group, 256 lanes and 32 groups make a tile), odd and mixed
sizes, conjugate pairs with k = 0 among them, planar and 3-D k, node counts
around the LDS chunks, one to six encodings, static and moving nodes.

Tolerances: mixed 1e-5 (FP32 phase of a reduced turn, ~1e-7 per term), FP64
1e-10.
"""
import numpy as np
import pytest
import scipy.sparse as sp

from test_gpu_signal import _nodes, _pod, descriptor_callable, rel_l2

pytestmark = pytest.mark.gpu

TOL = {"mixed": 1e-5, "f64": 1e-10}


def _samples(sizes, conj, planar, seed=3):
    """One long 'readout' (n, 1, 1) whose samples come in groups of equal t, shuffled."""
    rng = np.random.default_rng(seed)
    k, t = [], []
    for i, g in enumerate(sizes):
        kg = rng.uniform(-150.0, 150.0, (g, 3))
        if conj:
            kg[g // 2:] = -kg[:g // 2]
            if i == 0:
                kg[0] = kg[g // 2] = 0.0
        k.append(kg)
        t.append(np.full(g, 0.3 + 0.37 * i))
    k, t = np.concatenate(k), np.concatenate(t)
    if planar:
        k[:, 2] = 0.0
    p = rng.permutation(t.size)
    return tuple(np.ascontiguousarray(k[p, d].reshape(-1, 1, 1)) for d in range(3)), t[p].reshape(-1, 1, 1)


@pytest.mark.parametrize("moving", [False, True])
@pytest.mark.parametrize("sizes,conj,planar,n,v", [
    ([16] * 40, True, True, 1000, 1),          # 32 groups to a tile
    ([16] * 33 + [18] * 3, False, False, 127, 2),
    ([32] * 20, True, False, 129, 3),
    ([31] * 20, False, True, 1025, 4),
    ([2, 600, 17, 64, 513, 1, 33], False, False, 300, 1),
    ([128] * 5, True, True, 4097, 2),
    ([130] * 3, True, True, 15, 1),            # past the pair search's group size
    ([256, 255, 512, 511, 2, 2], False, False, 64, 6),
    ([1] * 70, False, False, 33, 1),           # every sample its own t
    ([64] * 3, True, True, 1, 1),
])
def test_groups(gpu, sizes, conj, planar, n, v, moving):
    import oracle
    from feelmri_amd import MRI

    kloc, t = _samples(sizes, conj, planar)
    r0, phi, T2, mxy, w = _nodes(n, v, 11)
    motion = None
    if moving:
        motion = _pod(n, seed=11)
        motion.update_timeshift(1.0)
    M = sp.diags(w)
    ref = oracle.Signal(0, M, kloc, t, r0, phi, T2, mxy, descriptor_callable(motion) if moving else None)
    errs = {p: rel_l2(MRI.Signal(0, M, kloc, t, r0, phi, T2, mxy, motion, precision=p, method="direct"), ref)
            for p in TOL}
    print(len(sizes), conj, planar, n, v, moving, {p: f"{e:.2e}" for p, e in errs.items()})
    assert all(errs[p] <= TOL[p] for p in TOL), errs
