"""The transforms at every length with a two-factor kernel (and lengths beside them that have none): 3D transforms of
unequal axes against numpy in FP64, and the z-plane kernels against the line passes bit for bit."""
import numpy as np
import pytest

import t9hip

pytestmark = pytest.mark.gpu

# every length along each axis; line counts that are no multiple of the 16 lines of a workgroup
DIMS = [(15, 16, 18), (16, 18, 15), (18, 15, 16), (20, 24, 25), (24, 25, 20), (25, 20, 24), (27, 30, 32), (30, 32, 27),
        (32, 27, 30), (36, 40, 45), (40, 45, 36), (45, 36, 40), (48, 50, 54), (50, 54, 48), (54, 48, 50), (60, 64, 72),
        (64, 72, 60), (72, 60, 64), (75, 80, 81), (80, 81, 75), (81, 75, 80), (90, 96, 100), (96, 100, 90),
        (100, 90, 96), (108, 120, 16), (120, 16, 108), (16, 108, 120), (128, 135, 15), (135, 15, 128), (15, 128, 135),
        (144, 150, 18), (150, 18, 144), (18, 144, 150), (160, 180, 15), (180, 15, 160), (15, 160, 180),
        (192, 15, 16), (15, 192, 16), (16, 15, 192), (125, 15, 16), (1, 2, 240), (3, 200, 5), (10, 12, 9)]


@pytest.mark.parametrize("prec", [t9hip.T9_FP32, t9hip.T9_FP64])
@pytest.mark.parametrize("dims", DIMS)
def test_fft3d_lengths(dims, prec):
    import torch
    rng = np.random.default_rng(sum(dims))
    x = rng.standard_normal(dims[::-1]) + 1j * rng.standard_normal(dims[::-1])
    x = x.astype(np.complex64 if prec == t9hip.T9_FP32 else np.complex128)
    # unit roundoff times the depth of the transform (log2 of the points, each level rounding a product and a sum)
    tol = (6e-8 if prec == t9hip.T9_FP32 else 1.2e-16) * (4 + np.log2(x.size))
    for sign in (-1, 1):
        ref = np.fft.fftn(x.astype(np.complex128)) if sign < 0 else np.fft.ifftn(x.astype(np.complex128)) * x.size
        y = torch.from_numpy(x).cuda()
        torch.cuda.synchronize()
        t9hip.fft3d(y.data_ptr(), *dims, prec, sign)
        err = np.linalg.norm(y.cpu().numpy() - ref) / np.linalg.norm(ref)
        assert err < tol, (sign, err, tol)


@pytest.mark.parametrize("K", [(36, 36, 24), (50, 50, 27), (60, 60, 32), (90, 90, 36), (100, 100, 45), (108, 108, 40)])
def test_plane_lengths_match_lines(K, monkeypatch):
    s = t9hip.System.water_box(216, 6, 18.643, 4, key="ewald\newald-cutoff 7.0\nvdwterm none\npme-grid %d %d %d\n"
                               "pme-order 5\nlist-buffer 1.0\npolar-eps 1e-6\n" % K)
    monkeypatch.delenv("T9HIP_FFT", raising=False)
    a = t9hip.Context(s, t9hip.T9_FP32).induce()
    monkeypatch.setenv("T9HIP_FFT", "lines")
    b = t9hip.Context(s, t9hip.T9_FP32).induce()
    assert a[2].iterations == b[2].iterations
    assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1])


@pytest.mark.parametrize("K", [60, 64])
def test_reciprocal_energy_is_not_scaled(K):
    """The FP32 reciprocal energy passes the weights and the transform twice.  Errors of single values cancel in it; what
    scales whole frequencies does not: 2.1e-7 (K = 60) with butterfly constants and weights of 24 bits, 0.8e-7 (K = 64) from
    the twiddles' own rounding where the influence function does not carry its inverse.  2e-8 is left, the charges'."""
    s = t9hip.System.water_box(4096, 16, 49.724, 21, key="ewald\newald-cutoff 7.0\npme-grid %d %d %d\npme-order 5\n"
                               "polar-eps 1e-6\nlist-buffer 1.0\npcg-precond\npcg-guess\nvdwterm none\n" % (K, K, K))
    e = {}
    for prec in (t9hip.T9_FP32, t9hip.T9_FP64):
        ctx = t9hip.Context(s, prec)
        e[prec] = ctx.energy()[0]["em_recip"]
        ctx.close()
    assert abs(e[t9hip.T9_FP32] / e[t9hip.T9_FP64] - 1) < 4e-8, e
