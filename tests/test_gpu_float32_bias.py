"""float32 evaluations have no error in common over their rows: the sine and
cosine instructions lose 3e-8 in modulus, which tables and row constants give
back, once for the phase that the detectors share and once for each detector
that rotates against it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _rows(seed, rows, duration, fs, dets, **kw):
    """Rows around the injection, where every bin of a sum counts alike."""
    from bilby_amd.configs import make_taylorf2_marginalised
    s = make_taylorf2_marginalised(n_draws=rows, seed=seed, duration=duration,
                                   sampling_frequency=fs, detectors=dets, distance=False, **kw)
    rng = np.random.default_rng(seed)
    for k, w in dict(mass_1=0.2, mass_2=0.2, theta_jn=0.1, phase=0.2, luminosity_distance=50.0,
                     ra=0.05, dec=0.03, psi=0.1, geocent_time=1e-3).items():
        s["draws"][k] = s["injection"][k] + w * rng.normal(size=rows)
    return s


@pytest.mark.parametrize("dets", [("H1",), ("H1", "L1", "V1"), ("H1", "L1", "V1", "K1")])
def test_inner_products(dets):
    """Relative error of <d|h> along itself, median over 500 rows: one row's is
    about 5e-8 / sqrt(1000 bins that count) = 2e-9, the data tables' rounding
    (in common) 2^-25 / sqrt(1000) = 1e-9.  Without the gain -3e-8 (one
    detector) to -5.5e-8 (four)."""
    from bilby_amd.likelihood import GravitationalWaveTransient
    s = _rows(3, 500, 8.0, 4096.0, dets, time=False, phase=False)
    lk = GravitationalWaveTransient(s["interferometers"], s["waveform_generator"],
                                    precision="fp32")
    lk.set_precision_escalation(0.0)
    aux = [lk.log_likelihood_ratio_batch(s["draws"], precision=p,
                                         return_inner_products=True)[1] for p in ("fp32", "fp64")]
    z = [a[:, 0] + 1j * a[:, 1] for a in aux]
    rel = (z[0] * z[1].conj()).real / np.abs(z[1]) ** 2 - 1.0
    assert np.abs(np.median(rel)) < 1e-8, np.median(rel)


@pytest.mark.parametrize("duration, fs, rows", [(8.0, 4096.0, 500),      # block projections
                                                (2.0, 2048.0, 1024)])    # a wavefront a row
def test_time_marginalised(duration, fs, rows):
    """lnL = ln I0(|<d|h>|) - <h|h> / 2 at the peak moves by about twice the
    relative error of <d|h> where both terms are of its size: -1.3e-7 without
    the gain.  Block projections have the rounding of the block functions in
    common (float32 tables, the same for every block and row), at most 2^-25 of
    their largest values: 3e-8 of <d|h>."""
    from bilby_amd.likelihood import GravitationalWaveTransient
    from tests.helpers import fixed_marginalised
    s = _rows(4, rows, duration, fs, ("H1", "L1", "V1"))
    priors = s["priors"].copy()
    lk = GravitationalWaveTransient(s["interferometers"], s["waveform_generator"],
                                    time_marginalization=True, phase_marginalization=True,
                                    priors=priors, precision="fp32")
    draws = fixed_marginalised(s["draws"], priors)
    out = [lk.log_likelihood_ratio_batch(draws, precision=p) for p in ("fp32", "fp64")]
    rel = out[0] / out[1] - 1.0
    assert np.abs(np.median(rel)) < 6e-8, np.median(rel)


def test_sine_gaussian_inner_products():
    """(limits as for TaylorF2; a burst's sum counts some 100 bins)"""
    from bilby_amd.configs import make_sine_gaussian_plain
    from bilby_amd.likelihood import GravitationalWaveTransient
    s = make_sine_gaussian_plain(n_draws=500, seed=3)
    rng = np.random.default_rng(3)
    for k, w in dict(frequency=3.0, Q=0.5, hrss=1e-23, ra=0.05, dec=0.03, psi=0.1,
                     geocent_time=1e-3).items():
        s["draws"][k] = s["injection"][k] + w * rng.normal(size=500)
    lk = GravitationalWaveTransient(s["interferometers"], s["waveform_generator"],
                                    precision="fp32")
    lk.set_precision_escalation(0.0)
    aux = [lk.log_likelihood_ratio_batch(s["draws"], precision=p,
                                         return_inner_products=True)[1] for p in ("fp32", "fp64")]
    z = [a[:, 0] + 1j * a[:, 1] for a in aux]
    rel = (z[0] * z[1].conj()).real / np.abs(z[1]) ** 2 - 1.0
    assert np.abs(np.median(rel)) < 2e-8, np.median(rel)
