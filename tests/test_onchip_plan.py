"""The plan of the one-launch CG (onchip_cg.hip), on the host: in the halo form a workgroup reads rows of
p that other workgroups wrote in the same iteration, and waits for `reach` workgroups on each side."""
import ctypes

import numpy as np
import pytest


def plan(vh, n, offsets, distinct=0, single=0, jacobi=0, cus=256):
    """(reach, first row of each workgroup and the end of the last); None: the system does not fit."""
    f = vh.lib().onchip_cg_plan
    f.argtypes = [ctypes.c_int, ctypes.c_int, ctypes.c_uint32, ctypes.c_uint32, ctypes.c_void_p, ctypes.c_uint32,
                  ctypes.c_uint32, ctypes.POINTER(ctypes.c_uint32), ctypes.c_void_p]
    off = np.array(sorted(offsets), np.int32)
    rows, reach = np.zeros(257, np.uint32), ctypes.c_uint32()
    wgs = f(single, jacobi, n, off.size, off.ctypes.data, distinct, cus, ctypes.byref(reach), rows.ctypes.data)
    return (reach.value, rows[:wgs + 1].astype(np.int64)) if wgs else None


def needed(n, offsets, rows):
    """Workgroups on each side that own a row of the system reached along a diagonal."""
    assert rows[0] == 0 and rows[-1] >= n and (np.diff(rows) >= 0).all()
    w = np.arange(rows.size - 1)
    end = np.minimum(rows[1:], n)
    most = 0
    for o in offsets:
        lo, hi = np.maximum(rows[:-1] + o, 0), np.minimum(end - 1 + o, n - 1)
        there = (lo <= hi) & (rows[:-1] < end)
        for at in (lo, hi):
            owner = np.searchsorted(rows, at[there], side="right") - 1
            most = max(most, int(np.abs(owner - w[there]).max(initial=0)))
    return most


def stencil(nx, ny, nz):
    o = [1, nx] + ([nx * ny] if nz > 1 else [])
    return [-k for k in o] + [0] + o


def check(vh, n, offsets, **kw):
    p = plan(vh, n, offsets, **kw)
    if p is None or p[0] == 0:
        return False
    assert p[0] >= needed(n, offsets, p[1]), (n, offsets, kw, p[0], needed(n, offsets, p[1]))
    return True


# Thin grids whose workgroups hold unequal numbers of chunks (product chunks no multiple of 256), where
# the reach in rows is many workgroups of the smaller kind.
THIN = [(1026, 27, 17), (1300, 19, 16), (1026, 41, 11), (1219, 63, 6), (1281, 62, 5), (1568, 63, 4), (1132, 37, 11),
        (1536, 30, 10), (1100, 43, 10)]


@pytest.mark.parametrize("grid", THIN + [(97, 83, 71), (128, 128, 128)])
@pytest.mark.parametrize("jacobi", [0, 1])
def test_halo_waits_for_all_it_reads(vh, grid, jacobi):
    n = int(np.prod(grid))
    halo = [check(vh, n, stencil(*grid), distinct=d, single=s, jacobi=jacobi) for d in (0, 1, 3) for s in (0, 1)]
    assert any(halo) or grid == (1568, 63, 4)  # 64 workgroups on each side: more than it waits for


def test_halo_waits_for_all_it_reads_over_ranges(vh):
    """Grids of all proportions and random bands, symmetric and one-sided, over the sizes that fit."""
    rng = np.random.default_rng(0)
    halo = 0
    for _ in range(6000):
        kind = rng.integers(4)
        if kind == 0:
            g = rng.integers([900, 2, 2], [2048, 64, 200])
        elif kind == 1:
            g = np.maximum(2, (np.exp(rng.uniform(np.log(2 ** 18), np.log(2 ** 22))) ** (1 / 3) * rng.uniform(0.6, 1.6, 3))).astype(int)
        if kind < 2:
            n, offsets = int(np.prod(g)), stencil(*map(int, g))
        else:
            n = int(np.exp(rng.uniform(np.log(2 ** 17), np.log(2 ** 22))))
            far = int(np.exp(rng.uniform(np.log(300), np.log(n / 4))))
            o = np.unique(rng.integers(1, max(2, min(far, 4000)), rng.integers(0, 3)))
            o = [int(k) for k in o] + [far]
            offsets = sorted(set([0] + o + ([-k for k in o] if kind == 2 else [])))
        halo += check(vh, n, offsets, distinct=int(rng.choice([0, 0, 1, 5])), single=int(rng.integers(2)),
                      jacobi=int(rng.integers(2)))
    assert halo > 1000
