"""Both neighbor lists against all pairs at the list radius: a few atoms, boxes of five cells per axis and of less (no
cells), boxes so sparse that 64 consecutive atoms spread over many cells, and so dense that the candidates take several
segments, batches of groups and row windows."""
import ctypes

import numpy as np
import pytest

import t9hip
from test_gpu_goldens import _brute_pairs
from test_gpu_vdw_types import noble_box

pytestmark = pytest.mark.gpu

KEY = "ewald\newald-cutoff %.1f\nvdw-cutoff %.1f\nlist-buffer 1.0\n"


@pytest.mark.parametrize("prec", [t9hip.T9_FP32, t9hip.T9_FP64])
@pytest.mark.parametrize("nmol,box,rm,rv", [(1, 18.0, 6.0, 6.0), (22, 18.0, 7.0, 5.0), (300, 20.8, 7.0, 5.0),
                                            (1500, 20.0, 9.0, 8.0), (1728, 33.0, 6.0, 6.5), (2000, 64.0, 5.0, 6.0),
                                            (700, 90.0, 6.0, 5.0)])
@pytest.mark.parametrize("mode", ["", "tiny"])
def test_lists_hold_all_pairs(nmol, box, rm, rv, mode, prec, monkeypatch):
    if mode:
        monkeypatch.setenv("T9HIP_LISTS", mode)
    s = t9hip.System.water_box(nmol, int(np.ceil(nmol ** (1 / 3) - 1e-9)), box, 11, key=KEY % (rm, rv))
    a = s.arrays()
    ctx = t9hip.Context(s, prec)
    parent, red = a["vdw_parent"].astype(int), a["vdw_red"]
    bond = a["xyz"] - a["xyz"][parent]
    bond -= box * np.rint(bond / box)
    sites = a["xyz"] + (red - 1.0)[:, None] * bond  # parent + red * bond, next to its atom
    for which, x, rc in ((0, a["xyz"], rm + 1.0), (1, sites, rv + 1.0)):
        have = {(int(i), int(k)) for i, k in ctx.nblist_pairs(which)}
        want, near = _brute_pairs(x, box, rc)
        assert have ^ want <= (near if prec == t9hip.T9_FP32 else set()), (which, len(have), len(want))


@pytest.mark.parametrize("prec", [t9hip.T9_FP32, t9hip.T9_FP64])
def test_lists_without_a_box(tmp_path, prec, monkeypatch):
    """No cells: every wave goes over all atoms, in one pass and in passes over 3 waves each."""
    s = noble_box(tmp_path, 2, 1000, 40.0, periodic=False)
    x = s.f64("xyz", (s.n, 3))
    r = np.sqrt(((x[:, None] - x[None]) ** 2).sum(-1))
    for mode in ("", "tiny"):
        monkeypatch.setenv("T9HIP_LISTS", mode)
        ctx = t9hip.Context(s, prec)
        for which, rc in ((0, 8.0), (1, 10.0)):
            have = {(int(i), int(k)) for i, k in ctx.nblist_pairs(which)}
            want = {(int(i), int(k)) for i, k in zip(*np.nonzero(np.triu(r < rc, 1)))}
            near = {(int(i), int(k)) for i, k in zip(*np.nonzero(np.triu(np.abs(r - rc) < 1e-5, 1)))}
            assert have ^ want <= near, (mode, which, len(have), len(want))
        ctx.close()


def test_a_list_too_long_takes_no_memory(tmp_path):
    """All pairs of 60,000 atoms exceed the list's 2^31 places: the error of the scan's counts, before room is made for
    its masks (1.1 GB) or for the list."""
    def free():  # of the HIP runtime the library is linked to
        a, b = ctypes.c_size_t(), ctypes.c_size_t()
        assert t9hip.lib().hipMemGetInfo(ctypes.byref(a), ctypes.byref(b)) == 0
        return a.value

    s = noble_box(tmp_path, 1, 60000, 160.0, periodic=False, cuts="")
    ctx = t9hip.Context(s, t9hip.T9_FP32)
    before = free()
    with pytest.raises(t9hip.T9Error) as err:
        ctx.nblist_build()
    assert err.value.code == t9hip.T9_ERR_LIST_OVERFLOW
    used = before - free()
    ctx.close()
    assert used < 400e6, used
