"""GPU check of block projections over batches larger than one pass of the
workspace (4096 rows in float32, 2048 in float64): rows on both sides of a pass
boundary have the values of smaller batches, and an evaluation counts once
where kernels are timed."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision, rows", [("fp32", 4096), ("fp32", 4097), ("fp32", 8200),
                                             ("fp64", 2049)])
def test_batches_past_one_pass(precision, rows):
    from bilby_amd._lib import LIB, check
    from bilby_amd.autotune import set_transform
    from bilby_amd.configs import make_taylorf2_marginalised
    from bilby_amd.likelihood import GravitationalWaveTransient
    from tests.helpers import fixed_marginalised
    s = make_taylorf2_marginalised(n_draws=rows, seed=21, duration=4.0, sampling_frequency=2048.0,
                                   detectors=("H1", "L1"), distance=False)
    priors = s["priors"].copy()
    lk = GravitationalWaveTransient(s["interferometers"], s["waveform_generator"],
                                    time_marginalization=True, phase_marginalization=True,
                                    priors=priors, precision=precision)
    set_transform(lk, 2)
    draws = fixed_marginalised(s["draws"], priors)
    check(LIB.gwl_event_timing(lk._event, 1))
    whole = lk.log_likelihood_ratio_batch(draws)
    ms, launches = ctypes.c_double(), ctypes.c_int64()
    check(LIB.gwl_event_timing_read(lk._event, ctypes.byref(ms), ctypes.byref(launches)))
    check(LIB.gwl_event_timing(lk._event, 0))
    assert launches.value == 1 and ms.value > 0.0
    parts = [lk.log_likelihood_ratio_batch({k: v[i:i + 1500] for k, v in draws.items()})
             for i in range(0, rows, 1500)]
    # float32 sums of a row do not depend on the batch; float64 ones are added
    # in another order where a row's work is cut differently
    assert np.max(np.abs(whole - np.concatenate(parts))) < 1e-9
