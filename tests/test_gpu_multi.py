"""GPU checks of the multi-event persistent launch (uneven batches): agrees
with the per-event path and the FP64 oracle, and a captured hipGraph replays
correctly with new rows between replays."""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def say(*a):
    print("[gpu-test]", *a, flush=True)
    sys.stdout.flush()


def _events():
    from bilby_amd.configs import make_uneven_events
    return make_uneven_events(n_events=5, seed=5, rows_range=(9, 70), durations=(4, 16, 32),
                              chi_range=0.8)


def _likelihoods(events):
    from bilby_amd.likelihood import GravitationalWaveTransient
    lks = []
    for ev in events:
        pri = ev["priors"].copy()
        lks.append(GravitationalWaveTransient(ev["interferometers"], ev["waveform_generator"],
                                              time_marginalization=True,
                                              distance_marginalization=True,
                                              phase_marginalization=True, priors=pri,
                                              precision="fp32"))
        ev["fixed_priors"] = pri
    return lks


def test_multi_event_matches_per_event_and_oracle():
    """Each event's rows through the persistent multi-event launch equal the
    per-event batched path to 1e-8 (only float64 summation order differs)
    and the FP64 oracle to 1e-3 (spot check of 3 rows per event)."""
    from bilby_amd.multi import MultiEventLikelihood
    from tests.helpers import draws_as_dicts, fixed_marginalised, oracle_from_setup
    say("multi-event vs per-event")
    events = _events()
    lks = _likelihoods(events)
    multi = MultiEventLikelihood(lks, [ev["n_rows"] for ev in events])
    single = []
    for e, (ev, lk) in enumerate(zip(events, lks)):
        d = fixed_marginalised(ev["draws"], ev["fixed_priors"])
        multi.set_parameters(e, d)
        single.append(lk.log_likelihood_ratio_batch(d))
    outs = [o.cpu().numpy() for o in multi.run()]
    for e in range(len(events)):
        assert np.max(np.abs(outs[e] - single[e])) < 1e-8, e
    for e, ev in enumerate(events[:3]):
        olk, _ = oracle_from_setup(ev)
        d = fixed_marginalised(ev["draws"], ev["fixed_priors"])
        ref = np.array([olk.log_likelihood_ratio(p) for p in draws_as_dicts(d, range(3))])
        say("event", e, "T", ev["interferometers"].duration, "max |dlnL|", np.max(np.abs(outs[e][:3] - ref)))
        assert np.max(np.abs(outs[e][:3] - ref)) < 1e-3


def test_multi_event_graph_replays():
    """A captured graph replayed three times, with new rows and row counts
    set between replays (and eager work and synchronisations in between),
    matches the eager per-event results every time."""
    import torch
    from bilby_amd.multi import MultiEventLikelihood
    from tests.helpers import fixed_marginalised
    say("multi-event graph replay")
    events = _events()
    lks = _likelihoods(events)
    multi = MultiEventLikelihood(lks, [ev["n_rows"] for ev in events])
    full = [fixed_marginalised(ev["draws"], ev["fixed_priors"]) for ev in events]
    for e in range(len(events)):
        multi.set_parameters(e, full[e])
    multi.capture()
    rng = np.random.default_rng(0)
    for rep in range(3):
        sub = []
        for e, ev in enumerate(events):
            n = int(rng.integers(1, ev["n_rows"] + 1))
            idx = rng.permutation(ev["n_rows"])[:n]
            d = {k: v[idx] for k, v in full[e].items()}
            multi.set_parameters(e, d)
            sub.append(d)
        outs = [o.cpu().numpy().copy() for o in multi.run()]
        eager = [lk.log_likelihood_ratio_batch(d) for lk, d in zip(lks, sub)]
        torch.cuda.synchronize()
        for e in range(len(events)):
            assert np.max(np.abs(outs[e] - eager[e])) < 1e-8, (rep, e)


def test_short_events_cross_between_forms():
    """Events of short segments take one wavefront a row from half as many rows as
    bins on, as in their own evaluation, and block projections below; the row
    counts of a captured graph cross that line between replays, next to an
    event that never does and one cut at the ISCO."""
    import torch
    from bilby_amd.configs import make_taylorf2_marginalised
    from bilby_amd.likelihood import GravitationalWaveTransient
    from bilby_amd.multi import MultiEventLikelihood
    from tests.helpers import fixed_marginalised
    say("multi-event: short segments")
    lks, draws = [], []
    for k, (duration, dets, rows, isco) in enumerate([
            (1.0, ("H1",), 601, None), (4.0, ("H1", "L1"), 33, None),
            (1.5, ("H1", "L1", "V1"), 770, "isco"), (1.0, ("H1", "L1"), 512, None)]):
        s = make_taylorf2_marginalised(n_draws=rows, seed=50 + k, duration=duration,
                                       sampling_frequency=2048.0, detectors=dets, distance=k == 3,
                                       taylorf2_termination=isco)
        priors = s["priors"].copy()
        lks.append(GravitationalWaveTransient(s["interferometers"], s["waveform_generator"],
                                              time_marginalization=True,
                                              distance_marginalization=k == 3,
                                              phase_marginalization=True, priors=priors))
        draws.append({key: np.array(v) for key, v in fixed_marginalised(s["draws"], priors).items()})
        draws[-1]["mass_1"][rows // 2] = -1.0
    full = [len(d["mass_1"]) for d in draws]
    multi = MultiEventLikelihood(lks, full)
    for captured in (False, True):
        if captured:
            multi.capture()
        for counts in (full, [511, 33, 767, 512], [601, 1, 768, 511], [3, 33, 770, 0], full):
            sub = [{key: v[len(v) - n:] for key, v in d.items()} for d, n in zip(draws, counts)]
            for e, n in enumerate(counts):
                if n:
                    multi.set_parameters(e, sub[e])
                else:
                    multi.rows[e] = 0
            outs = [o.cpu().numpy().copy() for o in multi.run()]
            torch.cuda.synchronize()
            for e, n in enumerate(counts):
                if n:
                    one = lks[e].log_likelihood_ratio_batch(sub[e])
                    # the same kernels' values, sums of blocks in another order
                    assert np.max(np.abs(outs[e][:n] - one)) < 1e-8, (captured, counts, e)
