"""Cartesian stacks whose lines and kz planes pair up about a centre take real
cosine / sine rows; the rest takes complex rows.  Both against the FP64 oracle
at the sizes where the pairing can go wrong: odd and even counts, one line or
plane, unpaired lines (partial Fourier), single-precision coordinates
(symmetric about 0 only), shuffled and repeated lines, shifted and rotated
stacks, row counts at the edges of the row blocks.

Tolerances: mixed 1e-4 (three bf16 products per real product keep ~2^-16 per
operand, FP32 accumulation), FP64 1e-10 (rounding of the phases).
"""
import numpy as np
import pytest
import scipy.sparse as sp

from feelmri_amd import trajectories

from test_gpu_signal import _nodes, _pod, descriptor_callable, rel_l2

pytestmark = pytest.mark.gpu

TOL = {"mixed": 1e-4, "f64": 1e-10}


def _stack(shape, form):
    kloc, t = trajectories.cartesian((0.24, 0.22, 0.2), shape, t_first=0.4)
    kx, ky, kz = (np.array(k) for k in kloc)
    rng = np.random.default_rng(5)
    if form == "partial":                       # the first third of the lines missing
        j0 = shape[1] // 3
        kx, ky, kz, t = (a[:, j0:] for a in (kx, ky, kz, np.asarray(t)))
    elif form == "float32":                     # coordinates rounded to float32
        ky, kz = ky.astype(np.float32).astype(np.float64), kz.astype(np.float32).astype(np.float64)
    elif form == "shuffled":
        p, q = rng.permutation(shape[1]), rng.permutation(shape[2])
        ky, kz = ky[:, p][:, :, q], kz[:, p][:, :, q]
    elif form == "repeated":                    # every line twice
        kx, ky, kz, t = (np.repeat(a, 2, axis=1) for a in (kx, ky, kz, np.asarray(t)))
    elif form == "shifted":
        ky, kz = ky + 13.7, kz - 5.3
    elif form == "rotated":                     # lines and planes mix y and z
        c, s = np.cos(0.3), np.sin(0.3)
        ky, kz = c * ky - s * kz, s * ky + c * kz
    elif form == "irregular":                   # no two offsets pair up
        ky = ky + rng.uniform(0, 2.0, shape[1])[None, :, None]
    return tuple(np.ascontiguousarray(a) for a in (kx, ky, kz)), np.ascontiguousarray(t)


@pytest.mark.parametrize("moving", [False, True])
@pytest.mark.parametrize("shape,v,form", [
    ((8, 96, 24), 4, "plain"), ((9, 33, 5), 3, "plain"), ((33, 1, 1), 1, "plain"), ((5, 2, 2), 1, "plain"),
    ((7, 31, 1), 2, "plain"), ((4, 129, 3), 1, "plain"), ((3, 64, 65), 1, "plain"), ((130, 17, 4), 1, "plain"),
    ((6, 96, 4), 1, "partial"), ((6, 64, 6), 2, "float32"), ((6, 40, 5), 2, "shuffled"), ((5, 24, 4), 1, "repeated"),
    ((6, 48, 7), 1, "shifted"), ((6, 48, 6), 1, "rotated"), ((6, 40, 4), 1, "irregular"),
])
def test_pairs(gpu, shape, v, form, moving):
    import oracle
    from feelmri_amd import MRI, device

    kloc, t = _stack(shape, form)
    assert device.analyse_trajectory(kloc, t, "auto")["method"] == "cartesian"
    n = 1203
    r0, phi, T2, mxy, w = _nodes(n, v, 7)
    motion = None
    if moving:
        motion = _pod(n, seed=7)
        motion.update_timeshift(2.0)
    M = sp.diags(w)
    ref = oracle.Signal(0, M, kloc, t, r0, phi, T2, mxy, descriptor_callable(motion) if moving else None)
    errs = {p: rel_l2(MRI.Signal(0, M, kloc, t, r0, phi, T2, mxy, motion, precision=p), ref) for p in TOL}
    print(shape, v, form, moving, {p: f"{e:.2e}" for p, e in errs.items()})
    assert all(errs[p] <= TOL[p] for p in TOL), errs
