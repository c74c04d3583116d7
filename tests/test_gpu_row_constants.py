"""Rows at the edges of the 64-row blocks that compute the row constants: each
batch gives the values its rows have in one-row batches, invalid rows included."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("detectors", [("H1",), ("H1", "L1", "V1", "K1")])
@pytest.mark.parametrize("rows", [1, 63, 64, 65, 129])
def test_batches_match_single_rows(rows, detectors):
    """float64: the same constants, and sums of 2048 terms below 2e3 that may be
    added in another order: sqrt(2048) 2^-53 2e3 = 1e-11, taken ten times."""
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
    invalid = rows // 2 if rows > 1 else None
    if invalid is not None:
        draws["mass_1"][invalid] = -1.0
    got = lk.log_likelihood_ratio_batch(draws)
    assert got.shape == (rows,)
    if invalid is not None:
        assert got[invalid] < -1e300
    pick = sorted({0, rows // 3, rows - 1} - {invalid})
    assert pick
    for r in pick:
        one = lk.log_likelihood_ratio_batch({k: v[r:r + 1] for k, v in draws.items()})
        # and as the last of 66 copies, past the first block of 64
        many = lk.log_likelihood_ratio_batch({k: np.repeat(v[r], 66) for k, v in draws.items()})
        assert abs(got[r] - one[0]) < 1e-10 and abs(got[r] - many[-1]) < 1e-10
