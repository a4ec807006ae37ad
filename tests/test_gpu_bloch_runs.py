"""Runs of like events in the Bloch integrator against the FP64 oracle: the
rotation kept over a run (hard pulses, gradient plateaus, delays) with dt that
varies by roundings, drifts out of the corrected range within a run, or steps;
runs across the 256-event chunks; one, two and three gradient axes; static
nodes and every instantiated mode count's edges; node counts around a block.

Tolerances: FP64 1e-10 as in the whole-sequence tests.  FP32: rounding the
angles (up to hundreds of radians over a run) leaves more than 1e-4 of a small
Mxy, so the bound is 4 times the error of the same steps in plain FP32: the
kernel rounds an angle where it is formed, where it is reduced and in the
hardware sine, the plain steps where it is formed.
"""
import numpy as np
import pytest

from feelmri_amd import sequences
from test_gpu_bloch_mass_pod import rel_l2

pytestmark = pytest.mark.gpu
GAMMA = sequences.GAMMA


def _events(T, seed):
    rng = np.random.default_rng(seed)
    rf, G, dt = np.zeros(T, complex), np.zeros((T, 3)), np.full(T, 0.01)
    axes = [(), (0,), (1,), (2,), (0, 2), (0, 1, 2)]
    i, kind = 0, 0
    while i < T:
        n = int(rng.choice([1, 2, 40, 300]))
        j = min(T, i + n)
        for a in axes[kind % 6]:
            G[i:j, a] = rng.normal() * 5
        if kind % 2 == 0:
            rf[i:j] = (rng.normal() + 1j * rng.normal()) * 1e-4
        base = rng.choice([0.0, 0.002, 0.01, 0.5])
        noise = [rng.normal(size=j - i) * 1e-15, np.arange(j - i) * 3e-13, np.zeros(j - i),
                 rng.choice([0.0, 1e-9], j - i)][kind % 4]
        dt[i:j] = base + noise
        i, kind = j, kind + 1
    return rf, G, dt


class _Steps:
    """Displacements of the steps in the order they are asked for (first: the start's)."""

    def __init__(self, disp):
        self.disp, self.i = disp, -1

    def __call__(self, t):
        self.i += 1
        return self.disp[max(self.i - 1, 0)]


def _plain_f32(r0, T1, T2, dB, M0, rf, G, dt, mxy, mz, disp):
    """The final state by the same steps in FP32."""
    f, c = np.float32, np.complex64
    r, x, z, dB = r0.astype(f), mxy.astype(c), mz.astype(f), dB.astype(f)
    rf, G, dt, gamma = rf.astype(c), G.astype(f), dt.astype(f), f(GAMMA)
    for i in range(1, dt.size):
        p = r if disp is None else r + disp[i - 1].astype(f)
        Bz = p @ G[i] + dB
        B = np.maximum(np.sqrt(Bz * Bz + f(abs(rf[i])) ** 2), f(1e-12))
        h = f(-0.5) * gamma * dt[i] * B
        a, b = np.cos(h) - f(1) * 1j * (Bz / B * np.sin(h)), -1j * (rf[i] / B) * np.sin(h)
        a, b = a.astype(c), b.astype(c)
        nx = f(2) * a.conj() * b * z + a.conj() ** 2 * x - b ** 2 * x.conj()
        nz = (abs(a) ** 2 - abs(b) ** 2) * z - f(2) * (a * b * x.conj()).real
        x = nx * np.exp(-dt[i] / T2.astype(f))
        z = nz + (f(M0) - nz) * -np.expm1(-dt[i] / T1.astype(f))
    return x, z


@pytest.mark.parametrize("n,R", [(1, 0), (256, 0), (257, 1), (63, 2), (70, 3), (70, 5), (70, 6), (70, 10), (70, 11),
                                 (300, 16)])
def test_bloch_runs(gpu, n, R):
    import torch

    from feelmri_amd import device
    import oracle

    T = 1100
    rng = np.random.default_rng(n + R)
    r0 = rng.uniform(-0.05, 0.05, (n, 3))
    T1, T2 = rng.uniform(0.3, 1500, n), rng.uniform(0.2, 100, n)
    dB = rng.normal(0, 20 / 42.58e6 * 1e3, n)
    mxy0, mz0 = (rng.normal(size=n) + 1j * rng.normal(size=n)) * 0.1, rng.uniform(0.5, 1.0, n)
    rf, G, dt = _events(T, 5 * n + R)
    motion = pod = disp = None
    if R:
        modes = (rng.normal(size=(3, R, n)) * 1e-3).astype(np.float32)
        coef = rng.normal(size=(T - 1, R + 3))
        coef[:, R:] *= 1e-3
        disp = np.einsum("crn,tr->tnc", modes.astype(np.float64), coef[:, :R]) + coef[:, None, R:]
        pod = _Steps(disp)
        motion = (torch.from_numpy(modes.reshape(3 * R, n)).to(gpu), torch.from_numpy(coef).to(gpu))
    wx, wz = oracle.solve_mri(r0, T1, T2, dB, 0.9, GAMMA, rf, G, dt, None, mxy0, mz0, pod, history=True)
    nodes = device.BlochNodes.from_arrays(r0, T1, T2, dB, device=gpu)
    ev = device.EventTable(rf, G, dt, device=gpu)
    x0, z0 = torch.from_numpy(mxy0).to(gpu), torch.from_numpy(mz0).to(gpu)
    px, pz = _plain_f32(r0, T1, T2, dB, 0.9, rf, G, dt, mxy0, mz0, disp)
    plain = max(rel_l2(px, wx[:, -1]), rel_l2(pz, wz[:, -1]))
    for prec, tol in (("f64", 1e-10), ("f32", 4 * plain)):
        fx, fz = device.bloch(nodes, ev, 0.9, GAMMA, x0, z0, precision=prec, motion=motion)
        hx, hz = device.bloch(nodes, ev, 0.9, GAMMA, x0, z0, precision=prec, motion=motion, history=True)
        e = [rel_l2(fx.cpu().numpy(), wx[:, -1]), rel_l2(fz.cpu().numpy(), wz[:, -1])]
        print(prec, n, R, " ".join(f"{v:.2e}" for v in e), f"bound {tol:.1e}")
        assert max(e) <= tol
        # the history's last column is the final state
        assert rel_l2(hx[:, -1].cpu().numpy(), fx.cpu().numpy()) <= 1e-7
        assert rel_l2(hz[:, -1].cpu().numpy(), fz.cpu().numpy()) <= 1e-7
        if prec == "f64":
            assert max(rel_l2(hx.cpu().numpy(), wx), rel_l2(hz.cpu().numpy(), wz)) <= tol


def test_bloch_non_finite_positions_stay_local(gpu):
    """A node at a non-finite position is NaN even where no gradient is on
    (0 times it is NaN); the other nodes of its wavefront are as without it."""
    import torch

    from feelmri_amd import device

    n, T = 130, 40
    rng = np.random.default_rng(2)
    r0 = rng.uniform(-0.05, 0.05, (n, 3))
    dB, one = rng.normal(0, 1e-4, n), np.ones(n)
    rf, G, dt = np.full(T, 1e-4 + 0j), np.zeros((T, 3)), np.full(T, 0.01)
    ev = device.EventTable(rf, G, dt, device=gpu)
    bad = r0.copy()
    bad[5, 1], bad[100, 2] = np.inf, np.nan
    for prec in ("f64", "f32"):
        out = []
        for r in (r0, bad):
            nodes = device.BlochNodes.from_arrays(r, 900 * one, 80 * one, dB, device=gpu)
            out.append(device.bloch(nodes, ev, 1.0, GAMMA, torch.zeros(n, dtype=torch.complex128, device=gpu),
                                    torch.ones(n, dtype=torch.float64, device=gpu), precision=prec))
        keep = np.ones(n, bool)
        keep[[5, 100]] = False
        for a, b in zip(*out):
            a, b = a.cpu().numpy(), b.cpu().numpy()
            assert np.array_equal(a[keep], b[keep]) and np.isnan(b[~keep]).all()
