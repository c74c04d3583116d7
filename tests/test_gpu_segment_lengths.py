"""GPU checks of the time transforms on segments whose number of bins is a
multiple of the transform length but no power of two, against the FP64 oracle
(one FFT of the whole segment): the tiled transform in both precisions, with
windows past one 512-point transform, for both source models and for several
events in one launch, and the transform under calibration marginalisation."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _limit(precision, ref):
    """float32: about eight factors (amplitude, phase factor, data, transform)
    of 2^-24 each, 5e-7 of inner products that are at most about 2 |lnL| + 1000
    here; float64 1e-8 of that scale leaves the oracle's own rounding room."""
    return (1e-3 + 1e-6 * np.abs(ref)) * (1.0 if precision == "fp32" else 1e-5)


def _setup(source, duration, fs, dets, half, rows):
    from bilby_amd.configs import make_sine_gaussian_plain, make_taylorf2_marginalised
    from bilby_amd.prior import Uniform
    if source == "taylorf2":
        s = make_taylorf2_marginalised(n_draws=rows, seed=41, duration=duration,
                                       sampling_frequency=fs, detectors=dets, chi_range=0.5,
                                       distance=False)
    else:
        s = make_sine_gaussian_plain(n_draws=rows, seed=41, duration=duration,
                                     sampling_frequency=fs, detectors=dets)
        s.update(time_marginalization=True, phase_marginalization=source == "phase")
        s["draws"]["time_jitter"] = np.zeros(rows)
        start = s["interferometers"].start_time
        s["draws"]["geocent_time"] = np.full(rows, start)
    centre = s["interferometers"].start_time + duration / 2
    s["priors"]["geocent_time"] = Uniform(centre - half, centre + half, name="geocent_time")
    return s


def _likelihood(s, precision, **kw):
    from bilby_amd.likelihood import GravitationalWaveTransient
    from tests.helpers import fixed_marginalised
    priors = s["priors"].copy()
    lk = GravitationalWaveTransient(s["interferometers"], s["waveform_generator"],
                                    time_marginalization=True,
                                    phase_marginalization=s["phase_marginalization"],
                                    priors=priors, precision=precision, **kw)
    return lk, fixed_marginalised(s["draws"], priors)


# duration, sampling rate, detectors, prior half width (s), rows
SHAPES = [
    (1.5, 2048.0, ("H1", "L1"), 0.1, 9),          # 1536 = 3 x 512 bins
    (6.0, 4096.0, ("H1", "L1", "V1"), 0.1, 5),    # 12288 = 24 x 512
    (3.0, 2048.0, ("H1",), 0.35, 4),              # 3072 = 3 x 1024, a window of 720
    (12.0, 4096.0, ("H1", "L1"), 5.9, 2),         # 24576 = 3 x 8192, a window of three slices
]


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("precision", ["fp32", "fp64"])
@pytest.mark.parametrize("source", ["taylorf2", "sinegaussian"])
def test_tiled_transform_matches_oracle(shape, precision, source):
    from bilby_amd.autotune import set_transform
    from tests.helpers import draws_as_dicts, oracle_from_setup
    duration, fs, dets, half, rows = shape
    s = _setup(source, duration, fs, dets, half, rows)
    lk, draws = _likelihood(s, precision)
    set_transform(lk, 1)
    out = lk.log_likelihood_ratio_batch(draws)
    olk, _ = oracle_from_setup(s)
    ref = np.array([olk.log_likelihood_ratio(p) for p in draws_as_dicts(draws, range(rows))])
    assert np.all(np.isfinite(ref))
    assert np.all(np.abs(out - ref) < _limit(precision, ref)), (out - ref, ref)


@pytest.mark.parametrize("precision", ["fp32", "fp64"])
def test_default_transform_matches_oracle(precision):
    """1536 bins: float64 has no block projections there (they take multiples
    of 1024 bins) and must agree with float32, which has."""
    from tests.helpers import draws_as_dicts, oracle_from_setup
    s = _setup("taylorf2", 1.5, 2048.0, ("H1", "L1"), 0.1, 9)
    lk, draws = _likelihood(s, precision)
    olk, _ = oracle_from_setup(s)
    ref = np.array([olk.log_likelihood_ratio(p) for p in draws_as_dicts(draws, range(9))])
    out = lk.log_likelihood_ratio_batch(draws)
    assert np.all(np.abs(out - ref) < _limit(precision, ref)), (out - ref, ref)


def test_several_events_match_oracle():
    """Sine-Gaussian events of 1536 and 12288 bins in one launch."""
    from bilby_amd.multi import MultiEventLikelihood
    from tests.helpers import draws_as_dicts, oracle_from_setup
    sets = [_setup("phase", 1.5, 2048.0, ("H1", "L1"), 0.1, 9),
            _setup("phase", 6.0, 4096.0, ("H1", "L1"), 0.1, 3)]
    pairs = [_likelihood(s, "fp32") for s in sets]
    multi = MultiEventLikelihood([lk for lk, _ in pairs], [9, 3])
    for e, (_, draws) in enumerate(pairs):
        multi.set_parameters(e, draws)
    outs = [o.cpu().numpy() for o in multi.run()]
    for s, (_, draws), out in zip(sets, pairs, outs):
        olk, _ = oracle_from_setup(s)
        ref = np.array([olk.log_likelihood_ratio(p)
                        for p in draws_as_dicts(draws, range(len(out)))])
        assert np.all(np.abs(out - ref) < _limit("fp32", ref)), (out - ref, ref)


@pytest.mark.parametrize("shape", [(3.0, 1024.0, ("H1", "L1"), 0.1, 4),     # 1536 bins
                                   (6.0, 2048.0, ("H1",), 0.1, 3)])         # 6144
@pytest.mark.parametrize("precision", ["fp32", "fp64"])
def test_calibration_with_time_matches_oracle(shape, precision, tmp_path):
    from bilby_amd import calibration as cal
    from oracle.calibration import OracleCalibrated
    from oracle.likelihood import OracleDetector, OracleEvent
    from tests.helpers import draws_as_dicts
    duration, fs, dets, half, rows = shape
    s = _setup("taylorf2", duration, fs, dets, half, rows)
    files = {}
    for ifo in s["interferometers"]:
        ifo.calibration_model = cal.CubicSpline("recalib_%s_" % ifo.name, 20.0, fs / 2, 5)
        s["priors"].update(cal.constant_uncertainty_spline_priors(0.1, 0.1, 20.0, fs / 2, 5,
                                                                  ifo.name))
        files[ifo.name] = str(tmp_path / ("%s.npz" % ifo.name))
    lk, draws = _likelihood(s, precision, calibration_marginalization=True,
                            number_of_response_curves=7, calibration_lookup_table=files)
    ifos = s["interferometers"]
    ev = OracleEvent([OracleDetector(i.name, i.frequency_array, i.frequency_domain_strain,
                                     i.power_spectral_density_array, i.frequency_mask)
                      for i in ifos], ifos.duration, ifos.sampling_frequency, ifos.start_time)
    olk = OracleCalibrated(ev, "taylorf2", lk.calibration_draws,
                           waveform_arguments=dict(s["waveform_generator"].waveform_arguments),
                           time_marginalization=True, phase_marginalization=True,
                           priors=dict(s["priors"]))
    ref = np.array([olk.log_likelihood_ratio(p) for p in draws_as_dicts(draws, range(rows))])
    out = lk.log_likelihood_ratio_batch(draws)
    assert np.all(np.abs(out - ref) < _limit(precision, ref)), (out - ref, ref)
