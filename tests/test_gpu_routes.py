"""Which kernels an evaluation runs (SignalPlan.route), and the ones that no other test's sizes reach: the
reduction of node splits by 8 threads an output (16 splits and more of few samples) behind every kernel that
splits, and the real-row Cartesian kernels of each number of row blocks, with the columns' rows staged and
not.  Sums against the FP64 oracle; tolerances of the paths: mixed 1e-4, FP64 1e-10."""
import numpy as np
import pytest
import scipy.sparse as sp

from feelmri_amd import trajectories
from test_gpu_signal import _nodes, rel_l2

pytestmark = pytest.mark.gpu
TOL = {"mixed": 1e-4, "f64": 1e-10}


def _spiral(samples, interleaves):
    return trajectories.spiral(0.24, 64, samples, interleaves, t_first=0.2)


def _stack(m, l, k, paired=True):
    """Lines and planes exactly symmetric about 0, or (not paired) at irregular places."""
    r = np.random.default_rng(m + l)
    kx = (np.arange(m) - m / 2) * 4.25
    ky, kz = ((np.arange(n) - (n - 1) / 2) * 4.5 for n in (l, k))
    if not paired:
        ky, kz = ky + r.uniform(0, 2.0, l), kz + r.uniform(0, 2.0, k)
    t = np.broadcast_to(np.linspace(0.5, 3.0, m)[:, None, None], (m, l, k))
    return [np.ascontiguousarray(np.broadcast_to(a, (m, l, k))) for a in
            (kx[:, None, None], ky[None, :, None], kz[None, None, :])], np.ascontiguousarray(t)


def _random(m, l, per_sample_t):
    r = np.random.default_rng(m * l)
    kloc = [r.uniform(-150.0, 150.0, (m, l, 1)) for _ in range(3)]
    t = r.uniform(0.5, 3.0, (m, l, 1)) if per_sample_t else \
        np.broadcast_to(np.linspace(0.5, 3.0, m)[:, None, None], (m, l, 1)).copy()
    return kloc, t


@pytest.mark.parametrize("kt,method,enc,modes,mixed,f64", [
    (_spiral(90, 32), "auto", 1, 0, "group_pairs", "group_pairs"),
    (_spiral(90, 31), "auto", 1, 0, "groups", "groups"),
    (_spiral(90, 16), "auto", 2, 3, "group_pairs", "group_pairs"),
    (_random(40, 15, False), "direct", 1, 0, "consecutive", "consecutive"),    # fewer than 16 samples a t
    (_random(40, 16, False), "direct", 1, 0, "groups", "groups"),
    (_random(40, 15, False), "direct", 1, 2, "groups", "groups"),              # moving: always
    (trajectories.radial(0.24, 150, 9, t_first=0.3), "auto", 1, 0, "lines", "runs"),
    (trajectories.radial(0.24, 100, 9, t_first=0.3), "auto", 1, 0, "runs", "runs"),
    (trajectories.radial(0.24, 150, 9, t_first=0.3), "auto", 1, 2, "groups", "groups"),
    (_stack(33, 64, 4), "auto", 2, 0, "cartesian_real", "cartesian_real"),
    (_stack(64, 64, 4, False), "auto", 2, 0, "cartesian", "cartesian"),
    (_stack(33, 64, 16), "auto", 2, 4, "cartesian_real", "cartesian_real"),
    (_stack(33, 64, 16, False), "auto", 2, 4, "cartesian", "cartesian"),
    (_stack(33, 64, 4), "auto", 5, 4, "groups", "groups"),                     # past the encodings of the GEMM
    # lines that the FP64 form finds further from a centre than its rounding
    (trajectories.cartesian((0.22,) * 3, (33, 128, 2), t_first=1.0), "auto", 1, 0, "cartesian_real", "cartesian"),
])
def test_routes(gpu, kt, method, enc, modes, mixed, f64):
    from feelmri_amd import device

    plan = device.SignalPlan(*kt, method=method)
    assert plan.route("mixed", 5000, enc, modes)[0] == mixed
    assert plan.route("f64", 5000, enc, modes)[0] == f64


def _check(kt, n, enc, precision, method, route, seed=3):
    import oracle
    from feelmri_amd import device

    r0, phi, T2, mxy, _ = _nodes(n, enc, seed)
    plan = device.SignalPlan(*kt, method=method)
    kind, splits = plan.route(precision, n, enc)
    assert kind == route
    nodes = device.SignalNodes.from_arrays(r0, phi, T2, mxy)
    got = plan.execute(nodes, precision=precision).cpu().numpy()
    want = oracle.Signal(0, sp.identity(n, format="csr"), *kt, r0, phi, T2, mxy).reshape(-1, enc)
    assert rel_l2(got, want) <= TOL[precision]
    return splits


@pytest.mark.parametrize("splits", [15, 16, 17, 23])
@pytest.mark.parametrize("kind,precision,method,route,per_split", [
    ("spoke", "f64", "direct", "runs", 2048), ("spoke", "mixed", "direct", "lines", None),
    ("short", "mixed", "direct", "runs", 2048), ("times", "f64", "direct", "consecutive", 2048),
    ("times", "mixed", "direct", "consecutive", 2048), ("group", "f64", "direct", "groups", 256),
    ("group", "mixed", "direct", "groups", 256), ("stack", "mixed", "auto", "cartesian", 128),
    ("stack", "f64", "auto", "cartesian", 128)])
def test_many_splits_of_few_samples(gpu, kind, precision, method, route, per_split, splits):
    kt = {"spoke": lambda: trajectories.radial(0.24, 131, 1, t_first=0.3),
          "short": lambda: trajectories.radial(0.24, 33, 1, t_first=0.3),
          "times": lambda: _random(7, 5, True), "group": lambda: _random(3, 17, False),
          "stack": lambda: _stack(3, 20, 2, False)}[kind]()
    n = (per_split or 256) * (splits - 1) + 3
    got = _check(kt, n, 1 if kind == "stack" else 1 + splits % 2, precision, method, route)
    assert got == splits if per_split else got >= 15


@pytest.mark.parametrize("lines", [16, 33, 64, 65, 90, 97, 127, 128, 130])
@pytest.mark.parametrize("precision", ["mixed", "f64"])
@pytest.mark.parametrize("m,k,enc", [
    (100, 1, 1),     # a column tile's readout rows do not fit the staging buffer
    (6, 30, 4),      # kz x encodings do not
    (64, 4, 1),      # they do
])
def test_real_rows_by_row_blocks(gpu, m, k, enc, precision, lines):
    _check(_stack(m, lines, k), 517, enc, precision, "auto", "cartesian_real")
