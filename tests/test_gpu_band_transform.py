"""GPU check of the block-projected window transform (gwl_band.hip) against
the FP64 oracle at the ends of its range: one step per block (512 bins), an
odd number of steps, a partial chunk, windows of a few bins and of all 512,
segments that are no power of two, one to four detectors, unequal masks, one
row and rows that do not fill a workgroup, split and unsplit work."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# duration, sampling rate, detectors, prior half width (s), rows
CASES = [
    (1.0, 1024.0, ("H1",), 0.05, 3),                 # 512 bins: one step a block
    (1.5, 2048.0, ("H1", "L1"), 0.1, 9),             # 1536 bins: three steps
    (4.0, 2048.0, ("H1", "L1", "V1"), 0.1, 17),      # one chunk
    (6.0, 4096.0, ("H1", "L1"), 0.1, 5),             # 12288 bins: three chunks
    (7.0, 1024.0, ("V1",), 0.2, 8),                  # 3584 bins: seven steps, padded to eight
    (8.0, 4096.0, ("H1", "L1", "V1", "K1"), 0.002, 33),  # a window of 14 bins
    (2.0, 2048.0, ("H1", "L1"), 0.1, 2),               # 2048 bins: two steps
    (8.0, 4096.0, ("H1", "L1", "V1"), 0.1237, 1),    # all 512 bins of the window, one row
]


# float64 takes whole steps in 256 blocks, multiples of 1024 bins; elsewhere (and
# where it is asked for, set_transform 2) it runs in tiles
RUNS = [(c, p) for p in ("fp32", "fp64") for c in CASES]


@pytest.mark.parametrize("case,precision", RUNS)
@pytest.mark.parametrize("split", [1, 64])
def test_window_transform_matches_oracle(case, precision, split):
    from bilby_amd.autotune import set_tile, set_transform
    from bilby_amd.configs import make_taylorf2_marginalised
    from bilby_amd.likelihood import GravitationalWaveTransient
    from bilby_amd.prior import Uniform
    from tests.helpers import draws_as_dicts, fixed_marginalised, oracle_from_setup
    duration, fs, dets, half, rows = case
    s = make_taylorf2_marginalised(n_draws=rows, seed=29, duration=duration,
                                   sampling_frequency=fs, detectors=dets, chi_range=0.5,
                                   distance=False)
    if len(dets) == 2:  # bins inside one detector's mask only
        s["interferometers"][1].minimum_frequency = 35.0
        s["interferometers"][0].maximum_frequency = fs / 2 - 60.0
    centre = s["priors"]["geocent_time"].minimum + 0.1
    s["priors"]["geocent_time"] = Uniform(centre - half, centre + half, name="geocent_time")
    priors = s["priors"].copy()
    lk = GravitationalWaveTransient(s["interferometers"], s["waveform_generator"],
                                    time_marginalization=True, phase_marginalization=True,
                                    priors=priors, precision=precision)
    draws = fixed_marginalised(s["draws"], priors)
    set_transform(lk, 2)
    set_tile(lk, 0, split)   # target wavefronts per CU: unsplit, and cut as far as it goes
    out = lk.log_likelihood_ratio_batch(draws)
    olk, _ = oracle_from_setup(s)
    ref = np.array([olk.log_likelihood_ratio(p) for p in draws_as_dicts(draws, range(rows))])
    # float32 integrand (2^-24 per factor) under a float64 sum: a few 1e-7 of
    # the inner products, which are of the order of |lnL| + rho^2 / 2 < 2000;
    # float64: 4e-14 (block functions, 512 window bins) and the sums' rounding
    tol = 1e-3 if precision == "fp32" else 1e-10
    assert np.max(np.abs(out - ref)) < tol, np.abs(out - ref).max()


@pytest.mark.parametrize("precision", ["fp32", "fp64"])
@pytest.mark.parametrize("rows", [6, 300])
def test_rows_cut_at_the_isco(precision, rows):
    """Supports that end in the first, a middle and the last group of blocks, past
    the band and below its start (no bin at all), mixed within workgroups, few
    rows (the steps are split) and more; alone, and as one of several events of
    which the other has no cut."""
    from bilby_amd.configs import make_taylorf2_marginalised
    from bilby_amd.likelihood import GravitationalWaveTransient
    from bilby_amd.multi import MultiEventLikelihood
    from tests.helpers import draws_as_dicts, fixed_marginalised, oracle_from_setup
    lks, draws, sets = [], [], []
    for termination in ("isco", None):
        s = make_taylorf2_marginalised(n_draws=rows, seed=33, duration=4.0,
                                       sampling_frequency=2048.0, detectors=("H1", "L1"),
                                       distance=False, taylorf2_termination=termination)
        # f_ISCO = 4397 Hz / (total mass): 14.7, 29, 129, 550, 970, 1465 Hz of 1024
        total = np.resize([300.0, 150.0, 34.0, 8.0, 4.53, 3.0], rows)
        s["draws"]["mass_1"], s["draws"]["mass_2"] = 0.55 * total, 0.45 * total
        priors = s["priors"].copy()
        lks.append(GravitationalWaveTransient(s["interferometers"], s["waveform_generator"],
                                              time_marginalization=True,
                                              phase_marginalization=True, priors=priors,
                                              precision=precision))
        draws.append(fixed_marginalised(s["draws"], priors))
        sets.append(s)
    out = lks[0].log_likelihood_ratio_batch(draws[0])
    olk, _ = oracle_from_setup(sets[0])
    pick = list(range(6)) + [rows - 1]
    ref = np.array([olk.log_likelihood_ratio(p) for p in draws_as_dicts(draws[0], pick)])
    # (tolerances as above)
    tol = 1e-3 if precision == "fp32" else 1e-10
    assert np.max(np.abs(out[pick] - ref)) < tol, np.abs(out[pick] - ref).max()
    if precision == "fp32":
        multi = MultiEventLikelihood(lks, [rows, rows])
        for e in range(2):
            multi.set_parameters(e, draws[e])
        got = [o.cpu().numpy() for o in multi.run()]
        for e in range(2):  # the same float32 sums, added in float64 in another order
            one = lks[e].log_likelihood_ratio_batch(draws[e])
            assert np.max(np.abs(got[e] - one)) < 1e-8
