"""Pencil segments of the y/z sweeps against the oracle and against each other
where the shape of the box or of the launch decides how they share waves."""
import numpy as np
import pytest

import hydropad_amd as hp
from helpers import FIELDS, NB, copy_state, rel_l1, to_hp_params
from hydropad_amd import ic
from oracle import HpCounters as OracleCounters

pytestmark = pytest.mark.gpu


def noisy_box(shape_interior, seed, amp, vamp):
    rng = np.random.default_rng(seed)
    shape = tuple(n + 2 * NB for n in shape_interior)
    st = {"p": 1.0 + amp * rng.random(shape), "rho": 1.0 + amp * rng.random(shape)}
    for k in ("vx", "vy", "vz"):
        st[k] = vamp * (rng.random(shape) - 0.5)
    return ic.periodic_fill({k: np.asfortranarray(v) for k, v in st.items()})


def run(st, P, d, seglen, precision="fp64", gforce=None):
    with hp.Box(st["p"].shape, precision) as box:
        box.set_params(to_hp_params(P, hp.HpParams))
        box.set_tiling(0, seglen, 0)
        box.upload(copy_state(st), gforce)
        box.reset_counters()
        box.ppmsolver(d)
        return box.counters(), box.download()


# 9, 16, 30 and 32 pencils share waves (7, 4, 2 and 2 segments each), 33 and 65 do not
@pytest.mark.parametrize("across", [(3, 3), (4, 4), (5, 6), (4, 8), (3, 11), (5, 13)], ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("n", [3, 50, 131])
def test_narrow_boxes(oracle, across, n):
    """Several segments in a wave: the bits of whole pencils and the oracle's
    values, and on a wild box (Courant number 4, some traced states negative)
    each interface counted once."""
    for d in (2, 3):
        shape = (across[0], n, across[1]) if d == 2 else (across[0], across[1], n)
        for wild in (False, True):
            st = noisy_box(shape, 3 + n + across[1], *((3.0, 2.0) if wild else (0.4, 0.4)))
            P = oracle.params(ngrid=n)
            oracle.timedet(P, oracle.speed(P, st), 4.0 if wild else 0.4, 1e30, 0.0)
            ref, cnt = copy_state(st), OracleCounters()
            oracle.ppmsolver(P, ref, d, counters=cnt)
            base = None
            for seglen in (4096, 0, 1, 2, 5, 24):
                c, out = run(st, P, d, seglen)
                base = base or (out, c.newton_iters_max)
                assert c.neg_state_clamps == cnt.neg_state_clamps, (shape, d, wild, seglen)
                assert c.newton_iters_max == base[1], (shape, d, wild, seglen)
                for k in FIELDS:
                    assert np.array_equal(out[k], base[0][k]), (shape, d, wild, seglen, k)
                    if not wild:
                        assert rel_l1(out[k], ref[k]) <= 1e-12, (shape, d, seglen, k, rel_l1(out[k], ref[k]))


@pytest.mark.parametrize("precision", ["fp64", "mixed", "fp64_exact"])
@pytest.mark.parametrize("gravity", [False, True], ids=["free", "gravity"])
@pytest.mark.parametrize("comoving", [False, True], ids=["static", "comoving"])
@pytest.mark.parametrize("gamma", [5.0 / 3.0, 1.66666667], ids=["5/3", "namelist"])
def test_segments_of_every_form(oracle, precision, gravity, comoving, gamma):
    """Pencils of 61 and 53 cells, whole (the window goes round 16 times) and
    in segments of 1, 7 and the launch's own length: on a mild box the oracle's
    values (relative L1 1e-12, mixed 2e-6) and the same bits, on a wild one
    (Courant number 4) the same bits and the oracle's count of clamped states,
    which there are, and, in the reference's order, of Newton iterations."""
    shape = (11, 61, 53)
    rng = np.random.default_rng(17)
    g = np.asfortranarray(0.05 * (rng.random((3,) + tuple(n + 2 * NB for n in shape)) - 0.5)) if gravity else None
    for wild in (False, True):
        st = noisy_box(shape, 23, *((3.0, 2.0) if wild else (0.4, 0.4)))
        P = oracle.params(gamma=gamma, ngrid=61)
        oracle.timedet(P, oracle.speed(P, st), 4.0 if wild else 0.4, 1e30, 0.0)
        if comoving:
            P.at, P.dat, P.rat, P.rdtath = 0.8, 0.5, 1.25, P.dt / 0.81
        for d in (2, 3):
            ref, cnt = copy_state(st), OracleCounters()
            oracle.ppmsolver(P, ref, d, gforce=g, counters=cnt)
            assert cnt.neg_state_clamps > 0 or not wild
            base = None
            for seglen in (4096, 0, 1, 7):
                c, out = run(st, P, d, seglen, precision, g)
                base = base or (c, out)
                if precision != "mixed":
                    assert c.neg_state_clamps == cnt.neg_state_clamps, (d, wild, seglen)
                if precision == "fp64_exact":
                    assert c.newton_iters_max == cnt.newton_iters_max, (d, wild, seglen)
                for name in ("neg_state_clamps", "newton_iters_max", "newton_nonconv"):
                    assert getattr(c, name) == getattr(base[0], name), (d, wild, seglen, name)
                for k in FIELDS:
                    assert np.array_equal(out[k], base[1][k]), (d, wild, seglen, k)
                    if not wild:
                        assert rel_l1(out[k], ref[k]) <= (2e-6 if precision == "mixed" else 1e-12), \
                            (d, seglen, k, rel_l1(out[k], ref[k]))
