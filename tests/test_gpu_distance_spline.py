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
