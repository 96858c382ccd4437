"""mdet_model_radius against the maximum of the two models' distance thresholds
found numerically from the published coefficient tables: an upper bound, at
most 1e-7 above it, over wide, narrow and degenerate ranges of log sizes."""
import math

import numpy as np
import pytest

import mdet_amd as M

LO, HI = math.log10(1500), math.log10(500000)


def _poly(which, x, y):
    # extended precision: the terms reach 1e8 where the sums are of order 10
    coef, ex = M.model_coefs(which)
    s = np.zeros(np.broadcast(x, y).shape, np.longdouble)
    for c, (a, b) in zip(coef, ex):
        s = s + np.longdouble(c) * x ** int(a) * y ** int(b)
    return s


def _maximum(xlo, xhi, T):
    """Largest (-T' - b) / c over xlo <= x <= y <= xhi by repeated grids."""
    floor = math.log(9.0)
    models = [(0, 1, max(T, floor))] + ([(2, 3, T)] if T < floor else [])
    best = -np.inf
    for b, c, t in models:
        x0, x1, y0, y1 = (np.longdouble(v) for v in (xlo, xhi, xlo, xhi))
        for _ in range(12):
            x = (x0 + (x1 - x0) * np.linspace(0, 1, 161, dtype=np.longdouble))[:, None]
            y = (y0 + (y1 - y0) * np.linspace(0, 1, 161, dtype=np.longdouble))[None, :]
            g = np.where(x <= y, (-t - _poly(b, x, y)) / _poly(c, x, y), -np.inf)
            i, j = np.unravel_index(int(np.argmax(g)), g.shape)
            best = max(best, float(g[i, j]))
            hx, hy = (x1 - x0) / 20, (y1 - y0) / 20
            x0, x1 = max(x[i, 0] - hx, np.longdouble(xlo)), min(x[i, 0] + hx, np.longdouble(xhi))
            y0, y1 = max(y[0, j] - hy, np.longdouble(xlo)), min(y[0, j] + hy, np.longdouble(xhi))
    return best


@pytest.mark.parametrize("cutoff", [0.7, 0.8, 0.9, 0.95, 0.98, 0.999])
@pytest.mark.parametrize("xlo,xhi", [(LO, HI), (LO, HI - 0.03), (LO + 0.2, HI - 0.7), (LO, LO + 1e-3),
                                     (LO + 1.0, HI), (HI - 1e-6, HI), (4.0, 4.0)])
def test_radius_is_within_its_tolerance_of_the_maximum(cutoff, xlo, xhi):
    T = math.log(1.0 / (1.0 - cutoff) - 1.0)
    want = _maximum(xlo, xhi, T)
    R = M.model_radius(xlo, xhi, cutoff)
    # the grids resolve a smooth maximum far below 1e-10; 1e-9 covers rounding
    assert want - 1e-9 <= R <= want + 1e-7 + 1e-9, (R, want)
