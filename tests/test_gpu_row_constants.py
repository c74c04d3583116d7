"""Rows at the edges of the 64-row blocks that compute the row constants: each
batch gives the values its rows have in one-row batches, invalid rows included."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("detectors", [("H1",), ("H1", "L1", "V1", "K1")])
@pytest.mark.parametrize("rows", [1, 63, 64, 65, 129])
def test_batches_match_single_rows(rows, detectors):
    """float64: the same constants, sums in another order, so 1e-12 of values
    up to a few hundred squared (float64 rounding of 4096 terms)."""
    from bilby_amd.configs import make_taylorf2_marginalised
    from bilby_amd.likelihood import GravitationalWaveTransient
    from tests.helpers import fixed_marginalised
    s = make_taylorf2_marginalised(n_draws=rows, seed=4, duration=4.0, sampling_frequency=1024.0,
                                   detectors=detectors)
    priors = s["priors"].copy()
    lk = GravitationalWaveTransient(
        s["interferometers"], s["waveform_generator"], time_marginalization=True,
        distance_marginalization=True, phase_marginalization=True, priors=priors,
        precision="fp64")
    draws = {k: np.array(v) for k, v in fixed_marginalised(s["draws"], priors).items()}
    draws["mass_1"][rows // 2] = -1.0
    got = lk.log_likelihood_ratio_batch(draws)
    assert got.shape == (rows,) and got[rows // 2] < -1e300
    for r in sorted({0, rows // 3, rows - 1} - {rows // 2}):
        one = lk.log_likelihood_ratio_batch({k: v[r:r + 1] for k, v in draws.items()})[0]
        assert abs(got[r] - one) <= 1e-12 * max(1.0, abs(one)) * 100
