"""The Mesher's force moments against the same trapezoid sum over the bilinear tiles in
extended precision: the workgroups' additions, some 4096 to an entry, go to 16 copies, so
that their roundings stay small beside the values' own.

Tolerance 8 * 2^-53 of the largest entry.  Of independent roundings, each 0.29 * 2^-53 RMS
of the partial sum it is made at, 4096 one after the other come to 19 * 2^-53 at the worst
(every partial sum as large as the result), 16 chains of 256, each of a sixteenth of the
result, to 1.2 * 2^-53; the values (a few ulp) and weights average over thousands of nodes."""
import ctypes as C

import numpy as np
import pytest

from bsalib_amd import abi, synth

pytestmark = pytest.mark.gpu
TOL = 8 * 2.0 ** -53
LD = np.longdouble


def _axis_weights(a, b, cells, points):
    """Weights of the cells + 1 nodes: sum over the trapezoid rule's points of their hats."""
    s = (points - 1) // cells
    w = np.full(points, LD(1.0))
    w[[0, -1]] = LD(0.5)
    out = np.zeros(cells + 1, dtype=LD)
    c = np.minimum(np.arange(points) // s, cells - 1)
    t = (np.arange(points) - c * s).astype(LD) / s
    np.add.at(out, c, w * (1 - t))
    np.add.at(out, c + 1, w * t)
    return out * (8 * np.arctan(LD(1.0)) * (LD(b) - LD(a)) / (points - 1))


def _level0(p, geom):
    """The axis nodes and the values on their square grid, [entry, j, i].  On an axis that
    is its own mirror image the second half is the mirrored first half, whose frequencies
    are the same to rounding only: the values at small |f| would show the difference."""
    x = [geom[0, 0]]
    for a, b, _, _, n in geom[geom[:, 2] == geom[0, 2], :5]:
        x += [b if i == n else a + i * ((b - a) / n) for i in range(1, int(n) + 1)]
    x = np.array(x)
    assert np.allclose(x, -x[::-1], rtol=0, atol=1e-12)
    f1, f2 = (v.ravel() for v in np.meshgrid(x, x))
    half = (f1.size + 1) // 2
    v, _ = abi.bfm_points(p, f1[:half], f2[:half], with_brm=False)
    v = np.concatenate([v, v[:, :f1.size - half][:, ::-1]], axis=1)
    return x, v.reshape(-1, x.size, x.size)


def _force_moments(p, M, level):
    geom, _ = M.tiles()
    dims, n = np.zeros((M.ntiles, 2), dtype=np.int32), C.c_int64(0)
    lv = np.full(M.ntiles, level, dtype=np.int32)
    ptr = lambda a: a.ctypes.data_as(C.POINTER(C.c_int32))  # noqa: E731
    assert abi.lib().bsahip_mesher_export(M.h, ptr(lv), 0, None, 0, ptr(dims), None, None, None,
                                          C.byref(n)) == 0
    x, lv0 = _level0(p, geom)
    out = np.zeros(M.nc, dtype=LD)
    first = {}                               # of two mirrored tiles the first stands for both
    for k, (a1, b1, a2, b2) in enumerate(geom[:, :4]):
        twin = tuple(np.round([-b1, -a1, -b2, -a2], 9))
        if twin in first:
            out += first[twin]
            continue
        n1, n2 = (int(v) for v in geom[k, 4:6])
        i0, j0 = np.abs(x - a1).argmin(), np.abs(x - a2).argmin()
        g1, g2 = (np.append(a + np.arange(m * level) * ((b - a) / (m * level)), b)
                  for a, b, m in ((a1, b1, n1), (a2, b2, n2)))
        f1, f2 = (v.ravel() for v in np.meshgrid(g1, g2))
        v, _ = abi.bfm_points(p, f1, f2, with_brm=False)
        v = v.reshape(-1, g2.size, g1.size)
        v[:, ::level, ::level] = lv0[:, j0:j0 + n2 + 1, i0:i0 + n1 + 1]
        w = np.outer(_axis_weights(a2, b2, n2 * level, int(dims[k, 1])),
                     _axis_weights(a1, b1, n1 * level, int(dims[k, 0])))
        one = (v.astype(LD) * w).sum(axis=(1, 2))
        first[tuple(np.round([a1, b1, a2, b2], 9))] = one
        out += one
    return out.astype(float), int(n.value)


@pytest.mark.parametrize("nn,seed", [(14, 0), (20, 1), (33, 2), (52, 3)])
def test_force_moments(gpu_lib, nn, seed):
    p = synth.tower(nn=nn, nm=2, comps=(1,), natf=np.array([0.2, 0.6]), xi=np.array([0.01, 0.015]),
                    nfreqs=33, df=0.125, seed=seed, u10=30.0)
    M = abi.Mesher(p, bkg_base_rfmnt=12 + 2 * seed, tile_cells=16)
    for level in (1, 2):
        want, points = _force_moments(p, M, level)
        assert points > 5e6
        runs = [M.run(levels=level), M.run(levels=level, per_tile=True),
                abi.mesher_run_batch([M], levels=[np.full(M.ntiles, level, np.int32)])[0]]
        for r in runs:
            assert np.abs(r["m3mf"] - want).max() <= TOL * np.abs(want).max(), (level, points)
    M.close()


def test_beyond_the_largest_number(gpu_lib):
    """A moment that exceeds the largest double is infinite, not NaN, on the Mesher's copies
    as on those of the FP64 contraction; the values it is made of are finite."""
    p = synth.tower(nn=14, nm=1, comps=(1,), natf=np.array([0.2]), xi=np.array([0.01]),
                    nfreqs=257, df=0.25, seed=0, u10=30.0)
    p.turb_scales = 0.05 * p.turb_scales                   # a wide peak at the origin
    cfg = dict(bkg_base_rfmnt=12, tile_cells=16)
    run = {"plan": lambda: abi.classic_run(p), "mesher": lambda: abi.Mesher(p, **cfg).run(levels=1)}
    base = {k: r()["m3mf"][0] for k, r in run.items()}
    peak = abi.bfm_points(p, np.zeros(1), np.zeros(1), with_brm=False)[0][0, 0]
    s = (1e308 / min(base.values())) ** (1 / 3)
    assert 0 < peak * s ** 3 < 2e307
    p.wfc = 4 ** (1 / 3) * s * p.wfc
    for k, r in run.items():
        assert np.isposinf(r()["m3mf"][0]), k
