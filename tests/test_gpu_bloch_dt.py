"""Steps whose dt departs by roundings from that of the decay factors at hand (FP64 form), against the
same steps in 80 bits: the departure's correction holds wherever the 256-event chunks cut the table."""
import numpy as np
import pytest

from feelmri_amd import sequences

pytestmark = pytest.mark.gpu
GAMMA = sequences.GAMMA
LD, CLD = np.longdouble, np.clongdouble


def _steps(r0, T1, T2, dB, rf, G, dt, mxy, mz, disp=None):
    r, x, z = r0.astype(LD), mxy.astype(CLD), mz.astype(LD)
    with np.errstate(divide="ignore"):
        R1, R2 = 1 / T1.astype(LD), 1 / T2.astype(LD)
    for i in range(1, dt.size):
        h = LD(dt[i])
        B = (r if disp is None else r + disp[i - 1].astype(LD)) @ G[i].astype(LD) + dB.astype(LD)
        q = CLD(rf[i])
        Bn = np.maximum(np.sqrt(B * B + abs(q) ** 2), LD(1e-12))
        th = -LD(GAMMA) * h * Bn / 2
        a, b = np.cos(th) - 1j * (B / Bn * np.sin(th)), -1j * (q / Bn * np.sin(th))
        nx = 2 * a.conj() * b * z + a.conj() ** 2 * x - b ** 2 * x.conj()
        nz = (abs(a) ** 2 - abs(b) ** 2) * z - 2 * (a * b * x.conj()).real
        e1 = np.exp(-h * R1)
        x, z = nx * np.exp(-h * R2), nz * e1 + (1 - e1)
    return x, z


def _run(gpu, r0, T1, T2, dB, rf, G, dt, mxy, mz):
    import torch

    from feelmri_amd import device

    nodes = device.BlochNodes.from_arrays(r0, T1, T2, dB)
    x, z = device.bloch(nodes, device.EventTable(rf, G, dt), 1.0, GAMMA, torch.tensor(mxy, device=gpu),
                        torch.tensor(mz, device=gpu), precision="f64")
    return x.cpu().numpy(), z.cpu().numpy()


def _inputs(n, T, seed=1):
    r = np.random.default_rng(seed)
    return (r.uniform(-0.1, 0.1, (n, 3)), r.normal(0, 1e-3, n), np.zeros(T, complex), np.zeros((T, 3)),
            r.normal(size=n) + 1j * r.normal(size=n), r.uniform(0.2, 1.0, n))


@pytest.mark.parametrize("shift", [0, 3, 250])
@pytest.mark.parametrize("rf_on", [False, True])
def test_departure_survives_the_end_of_a_chunk(gpu, shift, rf_on):
    """dt departs by 5e-13 ms once and then stays, over the end of a chunk (step 257); T2 of 1 us make a
    departure that is dropped worth 5e-10 a step, 1e-7 of the result.  Steps of exactly the same dt in
    80 bits; the FP64 steps round at 1e-16 each, 300 of them: bound 1e-12."""
    n, T = 70, 300
    r0, dB, rf, G, mxy, mz = _inputs(n, T)
    T1, T2 = np.full(n, 2e-3), np.full(n, 1e-3)
    dt = np.full(T, 1e-5)
    dt[0] = 0.0
    dt[2 + shift:] += 5e-13
    if rf_on:
        rf[:] = 1e-3 * (1 + 0.5j)
    want = _steps(r0, T1, T2, dB, rf, G, dt, mxy, mz)
    got = _run(gpu, r0, T1, T2, dB, rf, G, dt, mxy, mz)
    for g, w in zip(got, want):
        assert np.linalg.norm(g - w) <= 1e-12 * np.linalg.norm(w)


@pytest.mark.parametrize("zero", ["T1", "T2", "both", "tiny"])
def test_nodes_that_relax_at_once(gpu, zero):
    """T1 or T2 of 0 (or far below dt): the factor is exp(-inf) = 0 on every step, also where dt departs by
    roundings from the step before.  Other nodes of the wave keep their values (1e-12, as above)."""
    n, T = 70, 300
    r0, dB, rf, G, mxy, mz = _inputs(n, T)
    r = np.random.default_rng(3)
    T1, T2 = r.uniform(500, 1500, n), r.uniform(40, 100, n)
    short = 1e-9 if zero == "tiny" else 0.0
    if zero != "T2":
        T1[5] = short
    if zero != "T1":
        T2[[5, 64]] = short
    G[:] = np.repeat(r.normal(0, 5, (T // 50, 3)), 50, 0)
    rf[:] = 1e-3 * np.repeat(r.normal(size=T // 50), 50)
    dt = np.diff(1000.0 + np.arange(T) * 0.01, prepend=1000.0 - 0.01)
    want = _steps(r0, T1, T2, dB, rf, G, dt, mxy, mz)
    got = _run(gpu, r0, T1, T2, dB, rf, G, dt, mxy, mz)
    for g, w in zip(got, want):
        assert np.isfinite(g).all() and np.linalg.norm(g - w) <= 1e-12 * np.linalg.norm(w)


def test_fp32_recovery_does_not_depend_on_the_neighbours(gpu):
    """FP32 form: 1 - exp(-dt/T1) of a node is the same number whatever T1 the other nodes of its wave
    have, and Mz recovers by it: to 4 roundings of FP32 over 3 steps of dt/T1 = 1.3e-11."""
    import torch

    from feelmri_amd import device

    n, T = 64, 4
    r0, dB, rf, G, mxy, _ = _inputs(n, T)
    dt = np.array([0.0, 1.3e-8, 1.3e-8, 1.3e-8])
    mz = np.zeros(n)

    def run(T1):
        nodes = device.BlochNodes.from_arrays(r0, T1, np.full(n, 50.0), dB)
        return device.bloch(nodes, device.EventTable(rf, G, dt), 1.0, GAMMA, torch.tensor(mxy, device=gpu),
                            torch.tensor(mz, device=gpu), precision="f32")[1].cpu().numpy()

    T1 = np.full(n, 1000.0)
    alone = run(T1)
    T1[7] = 1.3e-8                     # exp(-1) for this node
    mixed = run(T1)
    other = np.arange(n) != 7
    assert np.array_equal(alone[other], mixed[other])
    assert np.abs(mixed[other] / 3.9e-11 - 1.0).max() <= 4 * 2.0 ** -24
    assert abs(mixed[7] - (1 - np.exp(-3.0))) <= 4 * 2.0 ** -24


@pytest.mark.parametrize("R", [0, 1, 3])
@pytest.mark.parametrize("precision", ["f64", "f32"])
@pytest.mark.parametrize("order", [(0, 128, 255), (255, 0, 64), (42, 43, 127), (128, 129, 0)])
def test_chunks_with_few_and_many_like_steps(gpu, order, precision, R):
    """Three chunks of 256 steps of which order[i] repeat the step before, spread over the chunk: the loop
    for single events and the one for runs follow each other in every order and carry dt, its departure
    and the state over.  FP64: 768 steps of up to 40 rad each in 80 bits, whose angle rounds at 40 x 1.1e-16 a
    step: 768 x 5e-15 = 4e-12.  FP32: 4 times the error of the same steps in plain FP32."""
    import torch

    from feelmri_amd import device
    from test_gpu_bloch_runs import _plain_f32

    n, T = 70, 769
    r0, dB, rf, G, mxy, mz = _inputs(n, T)
    r = np.random.default_rng(sum(order))
    T1, T2 = r.uniform(500, 1500, n), r.uniform(40, 100, n)
    like = np.zeros(T, bool)
    for c, k in enumerate(order):
        like[1 + 256 * c + np.sort(r.permutation(256)[:k])] = True
    like[1] = False
    dt = np.zeros(T)
    for i in range(1, T):
        if like[i]:
            rf[i], G[i], dt[i] = rf[i - 1], G[i - 1], dt[i - 1] + r.choice([0.0, 2e-15, -1e-13])
        else:
            rf[i] = r.choice([0.0, 1e-4]) * (r.normal() + 1j * r.normal())
            G[i] = r.normal(0, 5, 3) * (r.random(3) < 0.7) * (R == 0 or i % 3 == 0)
            dt[i] = r.choice([0.01, 0.01 + 1e-14, 0.004])
    motion, disp = None, None
    if R:
        modes = r.normal(0, 1e-3, (3 * R, n)).astype(np.float32)
        coef = np.concatenate([r.normal(size=(T - 1, R)), np.zeros((T - 1, 3))], axis=1)
        motion = (torch.tensor(modes, device=gpu), torch.tensor(coef, device=gpu))
        disp = np.einsum("crn,tr->tnc", modes.astype(float).reshape(3, R, n), coef[:, :R])
    nodes = device.BlochNodes.from_arrays(r0, T1, T2, dB)
    x, z = device.bloch(nodes, device.EventTable(rf, G, dt), 1.0, GAMMA, torch.tensor(mxy, device=gpu),
                        torch.tensor(mz, device=gpu), precision=precision, motion=motion)
    got = np.concatenate([x.cpu().numpy(), z.cpu().numpy()])
    want = np.concatenate(_steps(r0, T1, T2, dB, rf, G, dt, mxy, mz, disp))
    err = np.linalg.norm(got - want) / np.linalg.norm(want)
    if precision == "f64":
        assert err <= 4e-12
    else:
        plain = np.concatenate(_plain_f32(r0, T1, T2, dB, 1.0, rf, G, dt, mxy, mz, disp))
        assert err <= 4 * np.linalg.norm(plain - want) / np.linalg.norm(want)
