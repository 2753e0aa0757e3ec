"""The Mesher's quadrature kernel at the edges of its launch shapes: mode counts on
both sides of every template, BFM cells of one BRM cell up to 256, tile edges, and
cells cut into runs of rows.  The moments must equal the trapezoid-weighted sums of
the exported integrand (bsahip_mesher_export, another kernel), taken with math.fsum.

Tolerance 1e-12 of the largest entry: a tile's sum holds at most 257^2 terms, each
correct to a few ulp (1e-15 relative), accumulated over at most 257 + 257 / 4 chained
roundings, with terms that may cancel by some two digits."""
import ctypes as C
import math

import numpy as np
import pytest

from bsalib_amd import abi, synth

pytestmark = pytest.mark.gpu
TOL = 1e-12


def _mesher(nm, rfmnt, tile, brm_cells):
    p = synth.tower(nn=4, nm=nm, comps=(1, 3), natf=np.linspace(0.2, 3.0, nm),
                    xi=np.linspace(0.02, 0.05, nm), nfreqs=9, df=0.5, seed=nm)
    # a background zone that holds every peak: tiles of equal level-0 cells only
    return abi.Mesher(p, bkg_base_rfmnt=rfmnt, tile_cells=tile, bkg_peakw=8.0, brm_cells=brm_cells)


def _by_export(M, levels):
    geom, _ = M.tiles()
    x = M.export(levels=levels)
    out, at = [], 0
    for k, (na, nb) in enumerate(x["dims"]):
        v = x["val"][at:at + na * nb].reshape(nb, na, -1)
        at += na * nb
        wa, wb = np.ones(na), np.ones(nb)
        wa[[0, -1]] = wb[[0, -1]] = 0.5
        h1 = (geom[k, 1] - geom[k, 0]) / (na - 1)
        h2 = (geom[k, 3] - geom[k, 2]) / (nb - 1)
        w = np.outer(wb, wa) * (2 * np.pi * h1) * (2 * np.pi * h2)
        t = (v * w[:, :, None]).reshape(na * nb, -1)
        out.append([math.fsum(t[:, e]) for e in range(t.shape[1])] if t.shape[1] < 100
                   else np.sum(t.astype(np.longdouble), axis=0).astype(float))
    return np.array(out)


def _check(M, levels):
    ref = _by_export(M, levels)
    r = M.run(levels=levels, per_tile=True)
    assert np.abs(r["tile_m3mr"] - ref).max() < TOL * np.abs(ref).max()
    tot = ref.sum(axis=0)
    assert np.abs(r["m3mr"] - tot).max() < TOL * np.abs(tot).max()
    q = M.run(levels=levels)
    assert np.abs(q["m3mr"] - tot).max() < TOL * np.abs(tot).max()
    assert np.abs(q["m3mf"] - r["m3mf"]).max() < TOL * np.abs(r["m3mf"]).max()


@pytest.mark.parametrize("nm", [1, 2, 3, 4, 5, 8, 9, 10, 12, 13, 16, 17, 24, 25, 32])
def test_mode_counts(gpu_lib, nm):
    M = _mesher(nm, 5, 2, 8)
    _check(M, np.array([1, 2, 4, 8], dtype=np.int32))      # 8, 4, 2 and 1 BRM cells per BFM cell
    M.close()


@pytest.mark.parametrize("nm,rfmnt,tile,brm", [(3, 2, 1, 256), (4, 3, 2, 128), (6, 3, 1, 64),
                                               (11, 2, 1, 64), (3, 4, 3, 2), (1, 2, 1, 256)])
def test_long_cells_and_row_runs(gpu_lib, nm, rfmnt, tile, brm):
    M = _mesher(nm, rfmnt, tile, brm)
    _check(M, 1)
    M.close()


@pytest.mark.parametrize("only_diag", [False, True])
def test_mirrored_tiles_at_unequal_levels(gpu_lib, only_diag):
    """Tiles (f1, f2) and (-f1, -f2) are integrated once when their levels agree: the
    same levels on both, on one of them only, and a layout whose pre-peak gap is cut
    unevenly (tiles without a mirror image) must all give the exported integrand's
    sums, and the evaluation counts of every tile."""
    p = synth.tower(nn=5, nm=2, comps=(1, 3), natf=np.array([0.4, 1.5]),
                    xi=np.array([0.05, 0.04]), nfreqs=9, df=0.5, seed=4)
    M = abi.Mesher(p, bkg_base_rfmnt=4, tile_cells=2, bkg_peakw=0.15, only_diag=only_diag)
    geom, rule = M.tiles()
    key = {tuple(np.round(g[:4], 9)): k for k, g in enumerate(geom)}
    twin = [key.get(tuple(np.round([-g[1], -g[0], -g[3], -g[2]], 9)), -1) for g in geom]
    assert any(t < 0 for t in twin) and any(t >= 0 and t != k for k, t in enumerate(twin))
    rng = np.random.default_rng(0)
    same = rng.choice([1, 2, 4], size=M.ntiles).astype(np.int32)
    for k, t in enumerate(twin):
        if t > k:
            same[t] = same[k]
    for lv in (np.ones(M.ntiles, np.int32), same,
               rng.choice([1, 2, 4], size=M.ntiles).astype(np.int32)):
        _check(M, lv)
        n = (geom[:, 4] * lv + 1) * (geom[:, 5] * lv + 1) - (geom[:, 4] + 1) * (geom[:, 5] + 1)
        r = M.run(levels=lv)
        assert r["evals_post"] == int(n.sum())
        assert r["brm_points"] == int(np.sum(np.prod(M.export(levels=lv)["dims"].astype(np.int64),
                                                     axis=1)))
    M.close()


@pytest.mark.parametrize("only_diag", [False, True])
def test_tiles_alone(gpu_lib, only_diag):
    """bsahip_mesher_run_tiles asked for the tiles' moments only, with each of the other
    outputs left out in turn: every slot is the one of the call that takes them all, the
    slots of mirror images among them (1e-13: the order of the atomic sums varies)."""
    M = _mesher(3, 5, 2, 8) if not only_diag else abi.Mesher(
        synth.tower(nn=4, nm=3, comps=(1, 3), natf=np.linspace(0.2, 3.0, 3),
                    xi=np.linspace(0.02, 0.05, 3), nfreqs=9, df=0.5, seed=3),
        bkg_base_rfmnt=5, tile_cells=2, bkg_peakw=8.0, brm_cells=8, only_diag=True)
    geom, rule = M.tiles()
    twin = {tuple(np.round(g[:4], 9)) for g in geom}
    assert any(tuple(np.round([-g[1], -g[0], -g[3], -g[2]], 9)) in twin for g in geom)
    want = M.run(per_tile=True)
    assert np.abs(want["tile_m3mr"]).max(axis=1).min() > 0.0
    ptr = lambda a: None if a is None else a.ctypes.data_as(C.POINTER(C.c_double))  # noqa: E731
    for with_f, with_r in ((False, False), (True, False), (False, True)):
        tiles = np.full((M.ntiles, M.nc), np.nan)
        f = np.zeros(M.nc) if with_f else None
        r = np.zeros(M.nc) if with_r else None
        assert abi.lib().bsahip_mesher_run_tiles(M.h, None, ptr(tiles), ptr(f), ptr(r), None) == 0
        for k in range(M.ntiles):
            w = want["tile_m3mr"][k]
            assert np.abs(tiles[k] - w).max() <= 1e-13 * np.abs(w).max(), (k, with_f, with_r)
        for got, key in ((f, "m3mf"), (r, "m3mr")):
            if got is not None:
                assert np.abs(got - want[key]).max() <= 1e-13 * np.abs(want[key]).max()
    M.close()
