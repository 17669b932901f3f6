"""A planar shock tube under gravity over several steps: gas at rest beside the
tube's waves amplifies an ulp, so the bar is what an ulp does to the oracle."""
import numpy as np
import pytest

import hydropad_amd as hp
from helpers import FIELDS, copy_state, rel_l1
from hydropad_amd import ic

pytestmark = pytest.mark.gpu

N, STEPS = 24, 8


def oracle_run(oracle, st, g):
    P = oracle.params(ngrid=N)
    dt, t = oracle.timedet(P, oracle.speed(P, st), 0.8, 1e30, 0.0)
    oracle.evolve(P, st, 1, STEPS, 0.8, 1e30, t, gforce=g)
    return st


@pytest.mark.parametrize("precision", ["fp64", "fp64_exact"])
@pytest.mark.parametrize("axis", [0, 1, 2])
def test_gravity_tube_within_rounding(oracle, axis, precision):
    """Eight steps against the oracle.  Pressures and densities moved by at most
    an ulp at the start move the oracle's own result by 1e-8 in pressure and
    1e-6 in the transverse velocities; the device rounds differently in each of
    the 24 sweeps, so 24 times the response to one such change is allowed."""
    st = ic.sod(N, axis)
    shape = st["p"].shape
    g = ic.gaussian_gforce(shape)
    ref = oracle_run(oracle, copy_state(st), g)
    rng = np.random.default_rng(axis)
    response = dict.fromkeys(FIELDS, 0.0)
    for _ in range(3):
        near = copy_state(st)
        for k in ("p", "rho"):
            near[k] = np.asfortranarray(near[k] * (1.0 + 2.0 ** -52 * rng.integers(-1, 2, shape)))
        moved = oracle_run(oracle, ic.periodic_fill(near), g)
        response = {k: max(response[k], rel_l1(moved[k], ref[k])) for k in FIELDS}
    with hp.Box(shape, precision) as box:
        box.upload(copy_state(st), gforce=g)
        dt, t = box.timedet(box.speed(), 0.8)
        box.evolve(1, STEPS, 0.8, t, dt)
        out = box.download()
    for k in FIELDS:
        assert rel_l1(out[k], ref[k]) <= 24 * response[k], (k, rel_l1(out[k], ref[k]), response[k])
