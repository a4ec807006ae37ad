"""Sums over node splits where 8 threads share an output (many splits of few
samples): output counts that end inside a workgroup, one output, split counts
around the 16 that the rule asks for and that 8 threads do not share evenly,
and outputs past the rule's bound, against the FP64 oracle for the per-line
product (mixed), the direct sum and its readout runs (FP64).

Tolerances: those of the paths, mixed 1e-4 and FP64 1e-10.
"""
import pytest

from feelmri_amd import trajectories

from test_gpu_signal import _check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [256 * 15, 256 * 16 + 1, 256 * 17, 256 * 23 + 7])
@pytest.mark.parametrize("n_meas,n_lines,v", [(128, 1, 1), (131, 3, 1), (129, 2, 3), (512, 130, 1)])
def test_split_sums(gpu, n_meas, n_lines, v, n):
    kloc, t = trajectories.radial(0.24, n_meas, n_lines, t_first=0.3)
    _check(kloc, t, n=n, v=v, seed=n_meas + n, precisions=("mixed", "f64"))


@pytest.mark.parametrize("n", [500, 4099, 6000])
def test_split_sums_few_samples(gpu, n):
    kloc, t = trajectories.radial(0.24, 1, 1, t_first=0.3)
    _check(kloc, t, n=n, v=1, seed=n, precisions=("mixed", "f64"))
