"""The convolution virial of the z pass at every transform length (the two-factor lengths in registers, with and without
the inverse, and lengths of the Stockham pass), on a grid whose x-y plane is no whole number of workgroups: energy,
gradient and virial of the electrostatics against the FP64 oracle."""
import numpy as np
import pytest

import oracle
import t9hip

pytestmark = pytest.mark.gpu

LENGTHS = [16, 18, 20, 24, 25, 27, 30, 32, 36, 40, 45, 48, 50, 54, 60, 64, 72, 75, 80, 81, 90, 96, 100, 108, 120, 128, 135,
           144, 150, 160, 180, 192] + [10, 125, 200, 240]


@pytest.mark.parametrize("K3", LENGTHS)
def test_virial_against_oracle(K3):
    s = t9hip.System.water_box(64, 4, 13.0, 3, key="ewald\newald-cutoff 5.0\npme-grid 18 20 %d\npme-order 5\n"
                               "polar-eps 1e-9\nlist-buffer 0.5\npcg-precond\npcg-guess\nusolve-cutoff 4.5\n"
                               "vdwterm none\n" % K3)
    o = oracle.Oracle(s.arrays())
    eo, go, vo = o.energy(*o.induce()[:2])
    for prec in (t9hip.T9_FP64, t9hip.T9_FP32):
        ctx = t9hip.Context(s, prec)
        e, g, v = ctx.energy_terms(t9hip.TERM_ELEC)
        ctx.close()
        err = (abs(e["em"] + e["ep"] - eo["em"] - eo["ep"]) / abs(eo["em_recip"]),
               np.linalg.norm(g - go) / np.linalg.norm(go), np.linalg.norm(v - vo) / np.linalg.norm(vo))
        print(K3, prec, "%.1e %.1e %.1e" % err, flush=True)
        # sums of some thousand terms that each round by 6e-8 (1.1e-16); the gradient takes second derivatives of the
        # rounded grid, so its error grows as the square of the points per A
        tol = np.array([1e-6, 3e-6 * (1 + K3 / 40) ** 2, 1e-5]) if prec == t9hip.T9_FP32 else np.full(3, 1e-11)
        # odd lengths: the moduli of the two highest frequencies, +-(K - 1) / 2, differ (their rule takes the first for
        # -(K + 1) / 2), so the d and p dipoles of one complex grid mix in them by that much, and the oracle's two
        # grids do not: 1e-8 of the virial at 25 points, nothing at 45
        if K3 % 2 and K3 < 45:
            tol = np.maximum(tol, 1e-7)
        assert np.all(err < tol), (prec, err)
