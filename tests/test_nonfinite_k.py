"""Trajectories with an infinite or NaN coordinate: pairs and runs are found to a tolerance
relative to the largest |k|, which such a coordinate must not widen."""
import numpy as np
import pytest

from feelmri_amd import trajectories
from feelmri_amd.device import analyse_trajectory


def _random_groups(groups=40, size=32, seed=1):
    r = np.random.default_rng(seed)
    kloc = [r.uniform(-200.0, 200.0, (groups, size, 1)) for _ in range(3)]
    t = np.broadcast_to(np.linspace(0.5, 3.0, groups)[:, None, None], (groups, size, 1)).copy()
    return kloc, t


@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan])
def test_no_pairs_or_runs_from_a_coordinate_that_is_not_finite(value):
    kloc, t = _random_groups()
    kloc[1][7, 3, 0] = value
    a = analyse_trajectory(kloc, t, method="direct")
    assert a["conj_pack"] == 1 and a["n_runs"] == 0
    # curved lines, and spokes, whose runs are all linear without it
    for kl, tt in (trajectories.spiral(0.24, 64, 90, 31, t_first=0.2), trajectories.radial(0.24, 100, 7, t_first=0.3)):
        kl = [np.array(k) for k in kl]
        kl[0][20, 3, 0] = value
        assert analyse_trajectory(kl, tt, method="direct")["n_runs"] == 0
    tt = np.array(t)
    tt[5] = value
    assert analyse_trajectory(_random_groups()[0], tt, method="direct")["n_runs"] == 0


def _nodes(device, N, V, R, seed=4):
    import torch

    r = np.random.default_rng(seed)
    mxy = r.normal(size=(N, V)) + 1j * r.normal(size=(N, V))
    nodes = device.SignalNodes.from_arrays(r.uniform(-0.1, 0.1, (N, 3)), r.normal(0, 0.1, N), r.uniform(20, 80, N), mxy)
    modes = torch.tensor(r.normal(0, 1e-3, (3 * R, N)).astype(np.float32), device=nodes.packed.device) if R else None
    return nodes, modes


@pytest.mark.gpu
@pytest.mark.parametrize("moving", [False, True])
@pytest.mark.parametrize("precision", ["f64", "mixed"])
@pytest.mark.parametrize("kind", ["groups32", "groups20", "radial", "cartesian"])
def test_other_samples_keep_their_values(kind, precision, moving):
    """One coordinate made infinite: its samples are NaN, every other one is what it is with that
    coordinate finite (to the form's rounding: the route of the sum may differ)."""
    import torch

    from feelmri_amd import device

    if kind == "cartesian":
        kloc, t = trajectories.cartesian((0.2, 0.2, 0.05), (33, 18, 4), t_first=0.5)
    elif kind == "radial":
        kloc, t = trajectories.radial(0.24, 150, 9, t_first=0.3)
    else:
        kloc, t = _random_groups(40, int(kind[6:]))
    kloc = [np.array(k) for k in kloc]
    R = 3 if moving else 0
    nodes, modes = _nodes(device, 700, 2, R)

    def run(kl):
        plan = device.SignalPlan(kl, t)
        motion = None
        if moving:
            c = np.random.default_rng(2).normal(size=(plan.n_tgroups, R + 3)) * 1e-2
            motion = (modes, torch.tensor(c, device=plan.device))
        return plan.execute(nodes, precision=precision, motion=motion).cpu().numpy().reshape(t.shape + (2,))

    want = run(kloc)
    bad = np.zeros(t.shape, bool)
    if kind == "cartesian":
        bad[:, 5, :] = True          # a whole line, so that the stack still factorises
    else:
        bad[20, 3, 0] = True
    kloc[1][bad] = np.inf
    got = run(kloc)
    assert np.isnan(got[bad]).all()
    tol = 1e-12 if precision == "f64" else 2e-5
    assert np.linalg.norm(got[~bad] - want[~bad]) <= tol * np.linalg.norm(want[~bad])


@pytest.mark.gpu
@pytest.mark.parametrize("moving", [False, True])
@pytest.mark.parametrize("precision", ["f64", "mixed"])
@pytest.mark.parametrize("size", [20, 32])
@pytest.mark.parametrize("paired", [False, True])
def test_infinite_z_shows_where_kz_is_zero(size, precision, moving, paired):
    """kz z is 0 times infinity: a node with an infinite z makes every sample NaN, in a plane too."""
    import torch

    from feelmri_amd import device

    kloc, t = _random_groups(40, size)
    kloc[2][:] = 0.0
    if paired:
        for k in kloc:
            k[:, size // 2:] = -k[:, :size // 2]
    r = np.random.default_rng(8)
    N, R = 300, 2
    r0 = r.uniform(-0.1, 0.1, (N, 3))
    plan = device.SignalPlan(kloc, t, method="direct")
    motion = None
    if moving:
        motion = (torch.zeros((3 * R, N), dtype=torch.float32, device=plan.device),
                  torch.zeros((plan.n_tgroups, R + 3), dtype=torch.float64, device=plan.device))

    def run():
        nodes = device.SignalNodes.from_arrays(r0, np.zeros(N), np.full(N, 50.0), np.ones((N, 1), complex))
        return plan.execute(nodes, precision=precision, motion=motion).cpu().numpy()

    assert np.isfinite(run()).all()
    r0[123, 2] = np.inf
    assert np.isnan(run()).all()
