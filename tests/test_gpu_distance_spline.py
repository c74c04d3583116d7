"""GPU check of the distance table's interpolant (bucketed interval search,
tabled reciprocals) against the host evaluation of the same knots and
coefficients (binary search, Cox-de Boor): values on knots, between them, at
the ends of the bounding box and outside it, of both signs, for the smallest
spline and for dense ones."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("every", [0, 40, 3])
def test_interpolant_matches_the_host_evaluation(every):
    from bilby_amd._lib import LIB, check, dptr
    from bilby_amd.configs import make_taylorf2_marginalised
    from bilby_amd.likelihood import GravitationalWaveTransient
    s = make_taylorf2_marginalised(n_draws=600, seed=3, duration=4.0, sampling_frequency=2048.0,
                                   detectors=("H1", "L1"), phase=False, time=False)
    lk = GravitationalWaveTransient(s["interferometers"], s["waveform_generator"],
                                    distance_marginalization=True, priors=s["priors"].copy(),
                                    precision="fp64")
    rows = lk.rows_from_parameters(dict(s["draws"]))
    rows[:, 5] = lk._ref_dist           # the table is read at <d|h>, <h|h> themselves
    _, aux = lk.log_likelihood_ratio_batch(rows, return_inner_products=True)
    x, y = np.ascontiguousarray(aux[:, 0]), np.ascontiguousarray(aux[:, 2])
    assert x.min() < 0 < x.max()

    def knots(v):
        """Knots at every few of the values that occur, the outermost left out."""
        v = np.sort(v)[1:-1]
        inner = v[every:-every:every] if every else v[:0]
        return np.concatenate([[v[0]] * 4, inner, [v[-1]] * 4])

    tx, ty = knots(x), knots(y)
    nx, ny = len(tx) - 4, len(ty) - 4
    c = np.random.default_rng(8).normal(size=(nx, ny))
    bbox = np.array([tx[0], tx[-1], ty[0], ty[-1]])
    check(LIB.gwl_event_set_distance_spline(lk._event, nx, ny, dptr(tx), dptr(ty), dptr(c),
                                            dptr(bbox)), "gwl_event_set_distance_spline")
    out = lk.log_likelihood_ratio_batch(rows)
    ref = np.zeros(len(x))
    check(LIB.gwl_spline2d_eval_host(nx, ny, dptr(tx), dptr(ty), dptr(c), len(x), dptr(x), dptr(y),
                                     dptr(ref)), "gwl_spline2d_eval_host")
    inside = np.isfinite(ref)
    assert np.array_equal(np.isneginf(out), ~inside) and 0 < (~inside).sum() < 10
    # a basis value takes about ten roundings and so does each of the 16
    # products of two of them (all within [0, 1]) with its coefficient
    tol = 16 * 20 * np.finfo(float).eps * np.max(np.abs(c))
    assert np.max(np.abs(out[inside] - ref[inside])) < tol


@pytest.mark.parametrize("knots", [8, 800, 6000])
@pytest.mark.parametrize("precision", ["fp32", "fp64"])
def test_interpolant_of_the_time_marginalised_rows(knots, precision):
    """The table that a row's workgroup stages, and where the row spans more knots
    than it can hold (6000: 870 in float32, 1740 in float64), the table itself:
    lnL against the host evaluation at the transform's values, of both signs, with
    bins outside the table."""
    import ctypes
    import torch
    from scipy.special import logsumexp
    from bilby_amd import _lib
    from bilby_amd.abi import P_TIME_JITTER
    from bilby_amd._lib import LIB, check, dptr
    from bilby_amd.configs import make_taylorf2_marginalised
    from bilby_amd.likelihood import GravitationalWaveTransient
    from tests.helpers import fixed_marginalised
    n = 48
    s = make_taylorf2_marginalised(n_draws=n, seed=3, duration=4.0, sampling_frequency=2048.0,
                                   detectors=("H1", "L1"), phase=False)
    for k in ("mass_1", "mass_2", "ra", "dec", "psi", "theta_jn"):   # a third of the rows loud
        s["draws"][k][::3] = s["injection"][k]
    priors = s["priors"].copy()
    lk = GravitationalWaveTransient(s["interferometers"], s["waveform_generator"],
                                    time_marginalization=True, distance_marginalization=True,
                                    priors=priors, precision=precision)
    draws = fixed_marginalised(s["draws"], priors)
    rows = torch.from_numpy(lk.rows_from_parameters(draws)).to("cuda:0")
    j0, L, step = ctypes.c_int64(), ctypes.c_int32(), ctypes.c_double()
    check(LIB.gwl_event_time_window(lk._event, ctypes.byref(j0), ctypes.byref(L),
                                    ctypes.byref(step)))
    dh = torch.empty((n, L.value, 2), dtype=torch.float64, device="cuda:0")
    hh = torch.empty(n, dtype=torch.float64, device="cuda:0")
    check(LIB.gwl_eval_time_series(lk._event, ctypes.c_void_p(rows.data_ptr()), n, _lib.NPARAM,
                                   _lib.FP64, ctypes.c_void_p(dh.data_ptr()),
                                   ctypes.c_void_p(hh.data_ptr()), None))
    torch.cuda.synchronize()
    x, y = dh[:, :, 0].cpu().numpy(), hh.cpu().numpy()
    # a table narrower than the values, so that some bins lie outside
    lo, hi = 0.9 * x.min(), 0.9 * x.max()
    assert lo < 0 < hi

    def axis(a, b, m):
        return np.concatenate([[a] * 4, np.linspace(a, b, m + 2)[1:-1], [b] * 4])

    tx, ty = axis(lo, hi, knots), axis(0.5 * y.min(), 1.5 * y.max(), 6)
    nx, ny = len(tx) - 4, len(ty) - 4
    c = np.ascontiguousarray(np.sin(40.0 * np.arange(nx) / nx)[:, None]
                             + 0.1 * np.arange(ny)[None, :])
    bbox = np.array([lo, hi, ty[0], ty[-1]])
    check(LIB.gwl_event_set_distance_spline(lk._event, nx, ny, dptr(tx), dptr(ty), dptr(c),
                                            dptr(bbox)), "gwl_event_set_distance_spline")
    out = lk.log_likelihood_ratio_batch(draws)
    ref = np.zeros(x.size)
    xs, ys = np.ascontiguousarray(x.ravel()), np.repeat(y, L.value)
    check(LIB.gwl_spline2d_eval_host(nx, ny, dptr(tx), dptr(ty), dptr(c), x.size, dptr(xs),
                                     dptr(ys), dptr(ref)))
    prior = s["priors"]["geocent_time"]
    jitter = rows[:, P_TIME_JITTER].cpu().numpy() if lk.jitter_time else np.zeros(n)
    t = (lk.interferometers.start_time + (j0.value + np.arange(L.value) + 1) * step.value)[None, :] \
        + jitter[:, None]
    ref = np.where((t >= prior.minimum) & (t <= prior.maximum), ref.reshape(n, -1), -np.inf)
    want = logsumexp(ref, axis=1) + np.log(2.0 / 2048.0 / (prior.maximum - prior.minimum))
    assert np.all(np.isfinite(want)) and np.isneginf(ref).any()
    # the table's slope is below 40 / (hi - lo); float32 values are within 1e-6 of
    # the largest, and a value outside may come in: one of 400 of equal weight
    slope = 40.0 / (hi - lo)
    tol = slope * 1e-6 * np.abs(x).max() + 1e-4 if precision == "fp32" else 1e-9
    assert np.max(np.abs(out - want)) < tol, np.abs(out - want).max()
