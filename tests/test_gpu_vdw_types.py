"""vdW pairs of systems with few and with many vdW types: up to 16 types the pair parameters are read from a table in
LDS, beyond from memory."""
import numpy as np
import pytest

import oracle
import t9hip

pytestmark = pytest.mark.gpu


def noble_box(tmp_path, ntypes, natoms, box, periodic=True, cuts="mpole-cutoff 7.0\nvdw-cutoff 9.0\n"):
    """Atoms of `ntypes` vdW types on a jittered lattice, each with its own radius and well depth."""
    lines = [l for l in open(t9hip.PARAMS) if l.split() and l.split()[0] in
             ("forcefield", "vdwtype", "radiusrule", "radiustype", "radiussize", "epsilonrule")]
    for t in range(ntypes):
        lines.append(f'atom {t + 1} {t + 1} X{t} "type {t}" 18 39.9 0\n')
        lines.append(f"vdw {t + 1} {3.0 + 0.05 * t:.3f} {0.05 + 0.01 * t:.4f}\n")
        lines.append(f"multipole {t + 1} 0.0\n 0.0 0.0 0.0\n 0.0\n 0.0 0.0\n 0.0 0.0 0.0\n")
        lines.append(f"polarize {t + 1} 0.0 0.0\n")
    prm = tmp_path / "noble.prm"
    prm.write_text("".join(lines))
    rng = np.random.default_rng(5)
    side = int(np.ceil(natoms ** (1 / 3)))
    site = np.array([(i, j, k) for i in range(side) for j in range(side) for k in range(side)])[:natoms]
    xyz = (site + 0.5) * (box / side) + rng.uniform(-0.2, 0.2, (natoms, 3))
    out = [f"{natoms} noble box\n"] + ([f"{box} {box} {box} 90 90 90\n"] if periodic else [])
    for i, r in enumerate(xyz):
        out.append(f"{i + 1} X{i % ntypes} {r[0]:.8f} {r[1]:.8f} {r[2]:.8f} {i % ntypes + 1}\n")
    path = tmp_path / "noble.xyz"
    path.write_text("".join(out))
    return t9hip.System.from_files(str(path), str(prm), "vdwterm only\nlist-buffer 1.0\n" + cuts)


def pair_sizes(a):
    """Sums of the sizes that the rounding of the pair terms scales with: over the pairs the repulsive plus the
    attractive energy and r times the force, and per atom the same of the force (a pair term is the small difference of
    the two near the minimum, and a lattice site's net force that of its pairs)."""
    x, box, nj = a["xyz"], a["box"], int(a["njvdw"])
    d = x[:, None] - x[None]
    d -= box * np.rint(d / box)
    r = np.sqrt((d ** 2).sum(-1)) + 1e3 * np.eye(len(x))
    t = a["jvdw"][:, None] * nj + a["jvdw"][None]
    rm, eps = a["vdw_rmin"][t], a["vdw_epsmix"][t]
    near = r <= a["vdw_cut"]
    rho = r / rm
    t1, t2 = (1.07 / (rho + 0.07)) ** 7, 1.12 / (rho ** 7 + 0.12)
    energy = eps * t1 * (t2 + 2)
    force = eps / rm * 7 * t1 * ((t2 + 2) / (rho + 0.07) + rho ** 6 * t2 / (rho ** 7 + 0.12))
    return 0.5 * (near * energy).sum(), 0.5 * (near * force * r).sum(), (near * force).sum(1)


@pytest.mark.parametrize("ntypes", [1, 16, 17, 23])
@pytest.mark.parametrize("prec", [t9hip.T9_FP32, t9hip.T9_FP64])
def test_vdw_type_tables(tmp_path, ntypes, prec):
    s = noble_box(tmp_path, ntypes, 343, 26.0)
    e_ref, g_ref, v_ref = oracle.Oracle(s.arrays()).md_energy()
    assert s.scalar("njvdw") == ntypes
    ctx = t9hip.Context(s, prec)
    e, g, v = ctx.energy()
    # a pair term is a chain of about 30 operations, each rounded to 6e-8 (1.1e-16), unbiased: about
    # sqrt(30) = 5 roundings of its own size; the sums are FP64
    tol = 5 * (6e-8 if prec == t9hip.T9_FP32 else 1.1e-16) * 2
    size, _, force = pair_sizes(s.arrays())
    assert abs(e["evdw"] - e_ref["evdw"]) < tol * size + 1e-13 * size
    assert np.all(np.abs(g - g_ref).max(1) < tol * force + 1e-12 * force)
    assert np.abs(v - v_ref).max() < (tol + 1e-12) * 9.0 * force.sum()
    ctx.close()


def test_fp32_sums_are_not_biased(tmp_path):
    """Single pair terms round either way, so sums over 3e4 pairs and more agree with FP64 far below 24 bits, up to what
    the rounding of the buffering constants 0.12 and 1.12 and of the force's prefactor (one per pair of types) leaves:
    6e-8 of the sizes of the terms at most."""
    s = noble_box(tmp_path, 3, 343, 26.0)
    out = {}
    for prec in (t9hip.T9_FP32, t9hip.T9_FP64):
        ctx = t9hip.Context(s, prec)
        out[prec] = ctx.energy()
        ctx.close()
    (e, _, v), (e_ref, _, v_ref) = out[t9hip.T9_FP32], out[t9hip.T9_FP64]
    size, work, _ = pair_sizes(s.arrays())
    assert abs(e["evdw"] - e_ref["evdw"]) < 6e-8 * size
    assert abs(np.trace(v - v_ref)) < 6e-8 * work
