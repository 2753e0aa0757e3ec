"""The Mesher's quadrature kernel at the edges of its launch shapes: mode counts on
both sides of every template, BFM cells of one BRM cell up to 256, tile edges, and
cells cut into runs of rows.  The moments must equal the trapezoid-weighted sums of
the exported integrand (bsahip_mesher_export, another kernel), taken with math.fsum.

Tolerance 1e-12 of the largest entry: a tile's sum holds at most 257^2 terms, each
correct to a few ulp (1e-15 relative), accumulated over at most 257 + 257 / 4 chained
roundings, with terms that may cancel by some two digits."""
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
