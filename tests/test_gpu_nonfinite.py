"""States whose arithmetic leaves the normal numbers: the tracing that skips
vanishing terms ends where the one that forms them all does."""
import numpy as np
import pytest

import hydropad_amd as hp
from helpers import FIELDS, NB
from hydropad_amd import ic

pytestmark = pytest.mark.gpu

SHAPE = (43, 37, 45)


def underflowing(rng):
    """p rho below the smallest double: the Lagrangian sound speed is zero."""
    st = {"p": 10.0 ** rng.uniform(-300, -250, SHAPE), "rho": 10.0 ** rng.uniform(-150, -100, SHAPE)}
    for k in ("vx", "vy", "vz"):
        st[k] = 1e-80 * rng.uniform(-1, 1, SHAPE)
    return st, 0.3 / 39 / 1e-80


def poisoned(rng):
    """Noise with a NaN, both infinities, a zero and a negative value in every field."""
    st = {"p": 1.0 + rng.random(SHAPE), "rho": 1.0 + rng.random(SHAPE)}
    for k in ("vx", "vy", "vz"):
        st[k] = rng.uniform(-1, 1, SHAPE)
    for a in st.values():
        for v in (np.nan, np.inf, -np.inf, 0.0, -1.0):
            a[tuple(rng.integers(NB, n - NB) for n in SHAPE)] = v
    return st, 0.3 / 39


@pytest.mark.parametrize("make", [underflowing, poisoned])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("gamma", [5.0 / 3.0, 1.4], ids=["5/3", "1.4"])
def test_nan_cells_are_those_of_the_whole_tracing(make, precision, gamma):
    """A sweep without gravity turns the same cells NaN as one under a gravity
    that is zero everywhere, whose tracing always forms every term."""
    for seed in (1, 2):
        st, dt = make(np.random.default_rng(seed))
        st = ic.periodic_fill({k: np.asfortranarray(a) for k, a in st.items()})
        for d in (1, 2, 3):
            nan = []
            for g in (None, np.zeros((3,) + SHAPE, order="F")):
                with hp.Box(SHAPE, precision, gamma=gamma) as box:
                    P = box.params
                    P.dt = P.rdtath = dt
                    box.set_params(P)
                    box.upload(st, g)
                    box.ppmsolver(d)
                    out = box.download()
                nan.append(np.array([np.isnan(out[k][(slice(NB, -NB),) * 3]) for k in FIELDS]))
            assert np.array_equal(*nan), (seed, d, int((nan[0] != nan[1]).sum()), int(nan[1].sum()))
