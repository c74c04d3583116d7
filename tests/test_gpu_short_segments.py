"""GPU checks of the kernels that whole batches of short segments take (one
wavefront a row in float32, one workgroup a row in float64) against the tiled
float64 transform on every row, and the FP64 oracle on a few: the fewest bins,
numbers of bins that are no power of two, the largest segment, rows at the line
of the dispatch and ragged, one to four detectors, the ISCO cut, invalid rows."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# duration, sampling rate, detectors, prior half width (s), rows, ISCO cut, distance
CASES = [
    (0.5, 2048.0, ("H1",), 0.05, 257, False, False),              # 512 bins: one sub-sequence
    (1.5, 2048.0, ("H1", "L1"), 0.1, 769, False, False),          # 1536 bins: three
    (1.0, 2048.0, ("H1", "L1", "V1"), 0.1, 1024, True, True),
    (2.0, 2048.0, ("H1", "L1", "V1", "K1"), 0.2491, 1030, False, False),  # 512 window bins
    (4.0, 2048.0, ("H1", "L1", "V1"), 0.1, 2049, True, True),
    (4.0, 4096.0, ("H1", "L1"), 0.002, 4097, False, True),        # 8192 bins
]


@pytest.mark.parametrize("case", CASES)
def test_whole_batches_match_tiles_and_oracle(case):
    from bilby_amd.autotune import set_transform
    from bilby_amd.configs import make_taylorf2_marginalised
    from bilby_amd.likelihood import GravitationalWaveTransient
    from bilby_amd.prior import Uniform
    from tests.helpers import draws_as_dicts, fixed_marginalised, oracle_from_setup
    duration, fs, dets, half, rows, isco, distance = case
    s = make_taylorf2_marginalised(n_draws=rows, seed=37, duration=duration,
                                   sampling_frequency=fs, detectors=dets, chi_range=0.5,
                                   distance=distance, taylorf2_termination="isco" if isco else None)
    if len(dets) == 2:  # bins inside one detector's mask only
        s["interferometers"][1].minimum_frequency = 35.0
    centre = s["priors"]["geocent_time"].minimum + 0.1
    s["priors"]["geocent_time"] = Uniform(centre - half, centre + half, name="geocent_time")
    priors = s["priors"].copy()
    lk = GravitationalWaveTransient(s["interferometers"], s["waveform_generator"],
                                    time_marginalization=True, phase_marginalization=True,
                                    distance_marginalization=distance, priors=priors,
                                    precision="fp64")
    draws = {k: np.array(v) for k, v in fixed_marginalised(s["draws"], priors).items()}
    draws["mass_1"][5] = -1.0
    got = {p: lk.log_likelihood_ratio_batch(draws, precision=p) for p in ("fp32", "fp64")}
    set_transform(lk, 1)
    tiled = lk.log_likelihood_ratio_batch(draws, precision="fp64")
    set_transform(lk, 0)
    assert got["fp32"][5] == got["fp64"][5] == tiled[5] < -1e300
    keep = np.arange(rows) != 5
    # float32: 2^-24 per factor of the integrand, a few 1e-7 of inner products
    # below 2000; float64: the sums' rounding in another order
    tol = {"fp32": 1e-3, "fp64": 1e-9}
    for p in got:
        assert np.max(np.abs(got[p] - tiled)[keep]) < tol[p], p
    pick = [0, 1, 6, rows - 1]
    olk, _ = oracle_from_setup(s)
    ref = np.array([olk.log_likelihood_ratio(q) for q in draws_as_dicts(draws, pick)])
    for p in got:
        assert np.max(np.abs(got[p][pick] - ref)) < max(tol[p], 1e-8), p
