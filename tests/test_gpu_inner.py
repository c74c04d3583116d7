"""GPU check of the tabled TaylorF2 inner products (gwl_inner.hip) against the
FP64 oracle at the edges of its units of 1024 bins: less than one unit, a unit
that holds the Nyquist bin alone, bands that start and end inside units, the
ISCO cut, one to four detectors, one row and rows that do not fill a
workgroup."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# duration, sampling rate, detectors, rows, ISCO cut
CASES = [
    (1.0, 512.0, ("H1",), 1, False),                     # 257 bins
    (1.0, 2048.0, ("H1", "L1"), 3, False),               # 1025 bins: Nyquist in its own unit
    (5.0, 2048.0, ("H1", "L1", "V1"), 9, True),          # 5121 bins
    (8.0, 4096.0, ("H1", "L1", "V1", "K1"), 17, False),
]


@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_inner_products_match_oracle(case, precision):
    from bilby_amd.configs import make_taylorf2_marginalised
    from bilby_amd.likelihood import GravitationalWaveTransient
    from tests.helpers import draws_as_dicts, oracle_from_setup
    duration, fs, dets, rows, isco = case
    s = make_taylorf2_marginalised(n_draws=rows, seed=31, duration=duration,
                                   sampling_frequency=fs, detectors=dets, chi_range=0.5,
                                   time=False, distance=False, phase=False,
                                   taylorf2_termination="isco" if isco else None)
    if len(dets) > 1:  # bins inside one detector's mask only
        s["interferometers"][1].minimum_frequency = 35.0
        s["interferometers"][0].maximum_frequency = fs / 2 - 60.0
    lk = GravitationalWaveTransient(s["interferometers"], s["waveform_generator"],
                                    precision=precision)
    out = lk.log_likelihood_ratio_batch(s["draws"])
    olk, _ = oracle_from_setup(s)
    ref = np.array([olk.log_likelihood_ratio(p) for p in draws_as_dicts(s["draws"], range(rows))])
    # float64: sums of up to 5e4 terms of size |lnL| and below; float32: rows
    # past the escalation bound are float64, the others within it
    tol = 1e-10 * np.maximum(1.0, np.abs(ref)) if precision == "fp64" else 1e-3
    assert np.all(np.abs(out - ref) < tol), np.abs(out - ref).max()
    # a row's value does not depend on its slot or its partner
    again = lk.log_likelihood_ratio_batch({k: v[::-1].copy() for k, v in s["draws"].items()})
    assert np.array_equal(again[::-1], out)


@pytest.mark.parametrize("duration", [8.0, 32.0])
def test_prefix_sums_of_hh_are_rounded_once(duration):
    """<h|h> comes from per-event prefix sums, so their error would be that of
    every row.  Bound: the row's amplitude and the oracle's take about ten
    roundings each (1e-15, random over rows: the median of 40 is a few times
    below), the sums themselves one; rounded at each of 16384 steps and more they
    are 5e-15 and more off."""
    from bilby_amd.configs import make_taylorf2_marginalised
    from bilby_amd.likelihood import GravitationalWaveTransient
    from tests.helpers import draws_as_dicts, oracle_from_setup
    s = make_taylorf2_marginalised(n_draws=40, seed=6, duration=duration,
                                   sampling_frequency=4096.0, detectors=("H1",), time=False,
                                   distance=False, phase=False)
    lk = GravitationalWaveTransient(s["interferometers"], s["waveform_generator"],
                                    precision="fp64")
    _, aux = lk.log_likelihood_ratio_batch(s["draws"], return_inner_products=True)
    olk, _ = oracle_from_setup(s)
    hh = np.array([olk.plain_inner_products(p)[1]
                   for p in draws_as_dicts(s["draws"], range(40))])
    rel = aux[:, 2] / hh - 1.0
    assert np.abs(np.median(rel)) < 1e-15, (np.median(rel), np.abs(rel).max())


def test_escalated_rows_carry_the_float64_bits():
    """Without escalation the float32 error stays below the coefficient that
    selects rows, times Q = |<d|h>| + <h|h>, where that matters (Q above 1000: the
    selection starts at 4000); with it the selected rows are those past the
    tolerance, with float64's values, and every row is within 1e-3."""
    from bilby_amd.configs import make_taylorf2_marginalised
    from bilby_amd.likelihood import GravitationalWaveTransient
    s = make_taylorf2_marginalised(n_draws=4095, seed=5, duration=4.0, sampling_frequency=2048.0,
                                   detectors=("H1", "L1", "V1"), time=False, distance=False,
                                   phase=False)
    rng = np.random.default_rng(5)
    s["draws"]["luminosity_distance"] = np.exp(rng.uniform(np.log(30.0), np.log(2000.0), 4095))
    lk = GravitationalWaveTransient(s["interferometers"], s["waveform_generator"],
                                    precision="fp32")
    d = s["draws"]
    out64, aux64 = lk.log_likelihood_ratio_batch(d, precision="fp64", return_inner_products=True)
    lk.set_precision_escalation(0.0)
    raw32 = lk.log_likelihood_ratio_batch(d)
    q = np.hypot(aux64[:, 0], aux64[:, 1]) + aux64[:, 2]
    loud = q > 1000.0
    assert np.max((np.abs(raw32 - out64) / q)[loud]) < 2e-7
    lk.set_precision_escalation()
    out32, aux32 = lk.log_likelihood_ratio_batch(d, return_inner_products=True)
    sure, maybe = 2e-7 * q > 8e-4 * 1.01, 2e-7 * q > 8e-4 * 0.99
    assert 100 < np.sum(sure) <= lk.escalated_rows() <= np.sum(maybe) < 4000
    assert np.array_equal(out32[sure], out64[sure]) and np.array_equal(aux32[sure], aux64[sure])
    assert np.array_equal(out32[~maybe], raw32[~maybe])
    assert np.max(np.abs(out32 - out64)) < 1e-3
