"""The PME spreading against a direct sum in FP64: grid sizes that 8 divides and does not (the last tile of an axis 1 to 7
points wide), unequal axes, few atoms and several chunks of atoms per tile."""
import numpy as np
import pytest

import t9hip
from test_gpu_gather import dm5, m5, spline

pytestmark = pytest.mark.gpu


def d2m5(x):
    return spline(3, x) - 2 * spline(3, x - 1) + spline(3, x - 2)


def direct_grid(xyz, box, K, charge, dip, quad):
    """Grid of point multipoles (charge [n], dip [n,3], quad [n,3,3]) and the sum of the sizes of its terms."""
    out, size = np.zeros(K[::-1]), np.zeros(K[::-1])
    for a, x in enumerate(xyz):
        f = x / box
        f = f + 0.5 - np.floor(f + 0.5)
        idx, w = [], []
        for d in range(3):
            u = f[d] * K[d]
            t = u - np.floor(u) + 4 - np.arange(5)
            s = K[d] / box[d]
            idx.append((int(np.floor(u)) - 4 + np.arange(5)) % K[d])
            w.append((m5(t), dm5(t) * s, d2m5(t) * s * s))
        terms = [(charge[a], (0, 0, 0))]
        terms += [(dip[a, d], tuple(int(e == d) for e in range(3))) for d in range(3)]
        terms += [(quad[a, d, e], tuple(int(k == d) + int(k == e) for k in range(3))) for d in range(3)
                  for e in range(3)]
        at = np.ix_(idx[2], idx[1], idx[0])
        for c, (l, m, o) in terms:
            t = c * w[2][o][:, None, None] * w[1][m][None, :, None] * w[0][l][None, None, :]
            out[at] += t
            size[at] += np.abs(t)
    return out, size


@pytest.mark.parametrize("prec", [t9hip.T9_FP32, t9hip.T9_FP64])
@pytest.mark.parametrize("nmol,K,box", [(1, (16, 16, 16), 13.0), (3, (18, 20, 24), 13.0), (30, (25, 27, 30), 13.0),
                                        (64, (16, 36, 45), 13.0), (64, (50, 18, 20), 13.0), (216, (16, 18, 16), 18.643),
                                        (65, (15, 16, 18), 13.0)])
def test_spread_grids(nmol, K, box, prec):
    s = t9hip.System.water_box(nmol, int(np.ceil(nmol ** (1 / 3) - 1e-9)), box, 3,
                               key="ewald\newald-cutoff 5.0\npme-grid %d %d %d\npme-order 5\nlist-buffer 0.5\n"
                               "vdwterm none\n" % K)
    ctx = t9hip.Context(s, prec)
    n, xyz = s.n, s.f64("xyz", (s.n, 3))
    rng = np.random.default_rng(nmol)
    # a product of three weights and a source, each rounded, over the atoms of a point; weights of a fraction rounded
    # to 6e-8 of a cell vary by a few times their own size
    tol = 64 * (6e-8 if prec == t9hip.T9_FP32 else 1.2e-16 * max(K))
    # an axis below 16 takes the fixed-point kernel: each of the at most 20 contributions to a point is rounded to half
    # a quantum (2^-32, 2^-44)
    quantum = 20 * 0.5 * 2.0 ** (-32 if prec == t9hip.T9_FP32 else -44) if min(K) < 16 else 0.0
    L = np.full(3, box)
    ud, up = rng.standard_normal((2, n, 3))
    got = ctx.pme_grid_uind(ud, up)
    none = np.zeros(n), np.zeros((n, 3, 3))
    for part, u in ((0, ud), (1, up)):
        ref, size = direct_grid(xyz, L, K, none[0], u, none[1])
        assert np.all(np.abs(got[..., part] - ref) <= tol * (size + size.max() * 1e-2) + quantum), part
    got = ctx.pme_grid_mpole()
    p = ctx.rpole()
    quad = p[:, [4, 7, 8, 7, 5, 9, 8, 9, 6]].reshape(-1, 3, 3)
    ref, size = direct_grid(xyz, L, K, p[:, 0], p[:, 1:4], quad)
    assert np.all(np.abs(got[..., 0] - ref) <= tol * (size + size.max() * 1e-2) + quantum)
    assert not got[..., 1].any()
    ctx.close()


def test_fp32_sums_do_not_lose_bits():
    """The rounding of the terms is the same share of a point however many atoms reach it; that of their sum is not: adding
    N of them in 24 bits rounds N partial sums, each by 2^-24 / sqrt(3) of about sqrt(N / 2) terms, against sqrt(N) terms
    in the result: 3.5e-7 of it at 96 atoms per point, beside 1.7e-7 from the terms.  Added in 24 bits only 16 staged atoms
    at a time, of which 3 or 4 reach a point, it is 0.7e-7, and with the terms' 1.9e-7 or 1.1 times theirs.  Multipoles:
    the neutral molecules' terms cancel, so the sum rounds more of the result (3.8e-7 beside 2.8e-7)."""
    err = []
    for nmol in (30, 1500):
        s = t9hip.System.water_box(nmol, int(np.ceil(nmol ** (1 / 3) - 1e-9)), 20.0, 3,
                                   key="ewald\newald-cutoff 5.0\npme-grid 18 18 18\npme-order 5\nlist-buffer 0.5\n"
                                   "vdwterm none\n")
        u = np.random.default_rng(7).standard_normal((2, s.n, 3))
        grids = {}
        for prec in (t9hip.T9_FP32, t9hip.T9_FP64):
            ctx = t9hip.Context(s, prec)
            ctx.mpole_init()
            grids[prec] = (ctx.pme_grid_uind(*u), ctx.pme_grid_mpole())
            ctx.close()
        err.append([np.linalg.norm(a - b) / np.linalg.norm(b)
                    for a, b in zip(grids[t9hip.T9_FP32], grids[t9hip.T9_FP64])])
    assert err[1][0] < 1.25 * err[0][0] and err[1][1] < 1.5 * err[0][1], err


@pytest.mark.parametrize("K", [20, 36, 40])
def test_fp32_weights_are_not_biased(K):
    """The part of the FP32 error along the FP64 result, a common factor of all grid points or field components: single
    roundings (1.7e-7 of a value) cancel in it over the 3,600 and more values, that of a constant in the weights or
    of the points per A would not (20 and 40 points on 20 A are exact in 24 bits, 36 are 2.6e-8 off)."""
    s = t9hip.System.water_box(200, 6, 20.0, 3, key="ewald\newald-cutoff 5.0\npme-grid %d %d %d\npme-order 5\n"
                               "list-buffer 0.5\nvdwterm none\n" % (K, K, K))
    rng = np.random.default_rng(K)
    u, grid = rng.standard_normal((2, s.n, 3)), rng.standard_normal((K, K, K, 2))
    out = {}
    for prec in (t9hip.T9_FP32, t9hip.T9_FP64):
        ctx = t9hip.Context(s, prec)
        ctx.mpole_init()
        out[prec] = (ctx.pme_grid_uind(*u), np.array(ctx.pme_fphi_uind(grid)))
        ctx.close()
    for got, ref in zip(out[t9hip.T9_FP32], out[t9hip.T9_FP64]):
        factor = ((got - ref) * ref).sum() / (ref * ref).sum()
        # five standard deviations of 1.7e-7 / sqrt(3,600) = 3e-9
        assert abs(factor) < 1.5e-8, factor
