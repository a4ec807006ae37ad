"""The FP64 signal against the same sums in 80 bits: a form that replaces the plain evaluation (paired
lines and planes as real rows, conjugate pairs of samples, readout runs) may be no further from them than a
plain FP64 evaluation in numpy is, which rounds k', the products with the position and their sum."""
import numpy as np
import pytest

from feelmri_amd import trajectories

pytestmark = pytest.mark.gpu
LD = np.longdouble
PI = LD("3.14159265358979323846264338327950288")
PI_F = LD(np.float32(np.pi)) / PI


def _signal(kloc, t, pos_of, b, T2, phi, exact):
    """(S,) sums; pos_of(t): (N, 3) positions in 80 bits."""
    F = LD if exact else np.float64
    factor, two_pi = (PI_F, 2 * PI) if exact else (float(np.float32(np.pi)) / np.pi, 2 * np.pi)
    k = [np.asarray(a).ravel().astype(F) * factor for a in kloc]
    tt, out, key = np.asarray(t).ravel(), [], None
    for s in range(tt.size):
        if key != tt[s]:
            key = tt[s]
            pos = pos_of(key).astype(F).T
            c = b * np.exp(-F(key) / T2.astype(F))
            off = F(key) * phi.astype(F) / two_pi
        u = k[0][s] * pos[0] + k[1][s] * pos[1] + k[2][s] * pos[2] - off
        a = two_pi * (u - np.rint(u))
        out.append(((np.cos(a) - 1j * np.sin(a)) * c).sum())
    return np.array(out)


def _check(gpu, kloc, t, R=0, method="auto", n=300, seed=1):
    import torch

    from feelmri_amd import device

    r = np.random.default_rng(seed)
    d = r.normal(size=(n, 3))
    r0 = d / np.linalg.norm(d, axis=1, keepdims=True) * r.random((n, 1)) ** (1 / 3) * np.array([0.10, 0.08, 0.06])
    phi, T2 = r.normal(0, 0.2, n), r.uniform(20, 80, n)
    b = r.uniform(0.05, 0.15, n) * np.exp(0.3j * r.normal(size=n))
    plan = device.SignalPlan(kloc, t, method=method)
    nodes = device.SignalNodes.from_arrays(r0, phi, T2, b)
    motion, pos_of = None, lambda tt: r0.astype(LD)
    if R:
        modes = r.normal(0, 5e-4, (3 * R, n)).astype(np.float32)
        coef = np.concatenate([r.normal(size=(plan.n_tgroups, R)), np.zeros((plan.n_tgroups, 3))], axis=1)
        motion = (torch.tensor(modes, device=gpu), torch.tensor(coef, device=gpu))
        m = modes.astype(LD).reshape(3, R, n)
        row = {float(x): c for x, c in zip(plan.tgroup_t, coef)}
        pos_of = lambda tt: r0 + np.einsum("crn,r->nc", m, row[float(tt)][:R].astype(LD))  # noqa: E731
    got = plan.execute(nodes, precision="f64", motion=motion).cpu().numpy()[:, 0]
    want = _signal(kloc, t, pos_of, b, T2, phi, True)
    plain = _signal(kloc, t, pos_of, b, T2, phi, False)
    norm = np.linalg.norm(want.astype(complex))
    err, bound = (float(np.linalg.norm((x - want).astype(complex)) / norm) for x in (got, plain))
    print(f"error {err:.3g}, plain FP64 {bound:.3g}")
    assert err <= bound


@pytest.mark.parametrize("shape", [(61, 63, 5), (33, 128, 2), (32, 160, 1), (125, 60, 1), (6, 127, 31), (128, 24, 8),
                                   (17, 1, 9)])
def test_cartesian(gpu, shape):
    kloc, t = trajectories.cartesian((0.22, 0.22, 0.22), shape, t_first=1.0, t_readout=3.0)
    _check(gpu, kloc, t)


@pytest.mark.parametrize("shape", [(9, 65, 17), (20, 96, 9), (12, 128, 1), (8, 160, 4)])
def test_moving_cartesian(gpu, shape):
    kloc, t = trajectories.cartesian((0.22, 0.22, 0.06), shape, t_first=1.0, t_readout=3.0)
    _check(gpu, kloc, t, R=3)


def _spiral(m, l):
    fov, res = (0.24, 0.24, 0.24), (256, l, 1)
    T_ms = trajectories.spiral_stack(fov, res, density_exponent=2.0, dtype=np.float64)[2]
    kloc, t, _ = trajectories.spiral_stack(fov, res, oversampling=2, t_start=0.5, density_exponent=2.0,
                                           receiver_bw=(m // 2) / (T_ms * 1e-3), dtype=np.float64)
    return kloc, t


@pytest.mark.parametrize("moving", [False, True])
@pytest.mark.parametrize("m,l", [(300, 32), (200, 31), (160, 48), (90, 16)])
def test_spiral(gpu, m, l, moving):
    """Interleaves half a turn apart (an even number of them) pair up as k and -k to a rounding."""
    kloc, t = _spiral(m, l)
    _check(gpu, kloc, t, R=3 if moving else 0)


def test_pairs_in_three_dimensions(gpu):
    """Pairs k, -k + a rounding, with kz."""
    r = np.random.default_rng(6)
    kloc = [r.uniform(-250.0, 250.0, (60, 24, 1)) for _ in range(3)]
    for k in kloc:
        k[:, 12:] = -k[:, :12] * (1 + 2.0 ** -52 * r.integers(-1, 2, (60, 12, 1)))
    t = np.broadcast_to(np.linspace(0.5, 4.0, 60)[:, None, None], (60, 24, 1)).copy()
    _check(gpu, kloc, t, method="direct")


def test_stack_far_from_the_centre(gpu):
    """(A rotated stack is left out: its split into axes rounds before any form is taken.)"""
    (kx, ky, kz), t = trajectories.cartesian((0.22, 0.22, 0.22), (24, 48, 4), t_first=1.0)
    _check(gpu, (kx, ky + 1000.0, kz - 333.3), t)
