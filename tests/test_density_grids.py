"""2D densities on grids that take one or two points per lane and long or short chunks of terms:
a point's density does not depend on the grid it is part of."""
import numpy as np
import pytest

from test_cpdf import CASES_2D, _gpu_estimator, _load


# The sums differ in order only: with up to some 10^4 terms a point, each rounded at 2^-53 of the
# largest partial sum, and points that differ in the last bit, 1e-11 of the peak is ample.
@pytest.mark.gpu
@pytest.mark.parametrize("name", CASES_2D)
def test_a_point_is_alike_on_every_grid(name):
    rec = _load(name)
    est, s = _gpu_estimator(rec)
    g = rec["grids2d"][0]

    def density(xl, xh, xr, yl, yh, yr):
        if s.n == 2:
            return est.get_2D_pointwise_cpdf(xl, xh, xr, yl, yh, yr)
        return est.get_marginal_2D_pointwise_cpdf(g["i1"], g["i2"], xl, xh, xr, yl, yh, yr)

    rx, ry = (g["xhigh"] - g["xlow"]) / 52, (g["yhigh"] - g["ylow"]) / 52
    X, Y, Z = (np.asarray(a).reshape(-1) for a in density(g["xlow"], g["xhigh"], rx, g["ylow"], g["yhigh"], ry))
    assert X.size > 2048
    peak = np.max(np.abs(Z))
    for nx, ny in ((3, 2), (9, 7), (40, 40)):
        x, y, z = (np.asarray(a).reshape(-1)
                   for a in density(g["xlow"] + 5 * rx, g["xlow"] + (5 + nx) * rx, rx, g["ylow"] + 5 * ry,
                                    g["ylow"] + (5 + ny) * ry, ry))
        print(f"case {name}: {z.size} of {Z.size} points", flush=True)
        compared = 0
        for k in range(z.size):
            at = np.argmin(np.abs(X - x[k]) / rx + np.abs(Y - y[k]) / ry)
            # every grid's last column and row are its upper limits, which may lie off the others'
            if abs(X[at] - x[k]) < 1e-9 * rx and abs(Y[at] - y[k]) < 1e-9 * ry:
                assert abs(Z[at] - z[k]) <= 1e-11 * peak
                compared += 1
        assert compared >= nx * ny
    est.shutdown()
