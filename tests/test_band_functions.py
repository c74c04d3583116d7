"""CPU check of the block functions of the window transform: 16 products
reproduce the exponentials of every bin of a block at every bin of the window."""
import numpy as np
import pytest


# blocks, bins a block, window bins, largest error
@pytest.mark.parametrize("blocks, bins, window, limit", [
    (128, 4, 6, 1e-15),            # the smallest segment and window
    (128, 128, 420, 6e-11),        # 8 s at 4096 Hz, 0.2 s
    (128, 128, 512, 1.3e-9),
    (128, 1024, 420, 1.3e-10),     # 64 s: the error grows with the bins of a block
    (128, 1024, 512, 3e-9),        # (the worst point moves to its end)
    (256, 64, 420, 2e-15),         # float64: as many bins in twice the blocks
    (256, 512, 420, 4e-15),
    (256, 64, 512, 1.5e-14),
    (256, 512, 512, 4e-14),
])
def test_sum_of_products(blocks, bins, window, limit):
    from bilby_amd._lib import LIB, check, dptr
    u, v = np.zeros((bins, 16)), np.zeros((8, window, 2))
    check(LIB.gwl_band_functions_host(blocks, bins, window, dptr(u), dptr(v)))
    t = np.arange(bins) - 0.5 * (bins - 1)
    kappa = np.arange(window) - window // 2
    turns = np.longdouble(1) * t[:, None] * kappa[None, :] / (np.longdouble(blocks) * bins)
    two_pi = 2 * np.arctan2(np.longdouble(0), np.longdouble(-1))
    got_re = sum(u[:, p, None] * v[p // 2, :, 0] for p in range(0, 16, 2))
    got_im = -sum(u[:, p, None] * v[p // 2, :, 1] for p in range(1, 16, 2))
    err = np.hypot((got_re - np.cos(two_pi * turns)).astype(float),
                   (got_im + np.sin(two_pi * turns)).astype(float))
    assert err.max() < limit, err.max()
