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


def run(st, P, d, seglen, precision="fp64"):
    with hp.Box(st["p"].shape, precision) as box:
        box.set_params(to_hp_params(P, hp.HpParams))
        box.set_tiling(0, seglen, 0)
        box.upload(copy_state(st))
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
