"""Bispectra of selected triples on the grid and at points at the edges of their tiles:
half grids around 16 and 32 points, one mode up to more than 32 (the point kernel's last
tile, then the general path), contractions of one padded chunk and more, one point and
many, zero and repeated frequencies.

Against oracle.classic_factorised and oracle.msh_points; tolerance 1e-12 of the largest
entry: sums of 3 * 200 products of three factors, each correct to a few ulp, and response
factors of damped modes (relative error of a few ulp over twice the damping ratio)."""
import numpy as np
import pytest

from bsalib_amd import abi, synth
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _tower(nn, nm, nfh, comps, seed=3):
    return synth.tower(nn=nn, nm=nm, comps=comps, natf=np.linspace(0.2, 3.0, nm), nfreqs=nfh,
                       df=4.0 / nfh, seed=seed)


def _rel(a, b):
    return np.abs(a - b).max() / np.abs(b).max()


@pytest.mark.parametrize("exact", [False, True])
@pytest.mark.parametrize("nn,nm,nfh,comps", [(1, 1, 2, (1,)), (7, 2, 15, (1, 3)), (40, 3, 16, (1,)),
                                             (9, 3, 17, (1, 2, 3)), (33, 5, 32, (3,)),
                                             (200, 4, 33, (1, 2, 3)), (16, 6, 50, (1,))])
def test_selected(gpu_lib, nn, nm, nfh, comps, exact):
    p = _tower(nn, nm, nfh, comps)
    nf = 2 * nfh - 1
    o = O.classic_factorised(p, truncate=not exact, want_bisp=True)
    want = {"bisp_f": o["bfm"], "bisp_r": o["brm"]}
    sel = sorted({1, nm ** 3, 1 + nm ** 3 // 2, 1 + nm ** 3 // 3})
    r = abi.classic_bispectra_sel(p, sel, exact=exact)
    full = abi.classic_spectra(p, exact=exact)
    for k in ("bisp_f", "bisp_r"):
        w = want[k].reshape(nm ** 3, nf, nf, order="F")
        for c, s in enumerate(sel):
            assert _rel(r[k][:, :, c], w[s - 1]) < 1e-12, (k, s)
            assert np.array_equal(r[k][:, :, c], full[k][:, :, s - 1])
        assert _rel(full[k], np.moveaxis(w, 0, 2)) < 1e-12


@pytest.mark.parametrize("nn,nm,comps,npts", [(1, 1, (1,), 1), (9, 3, (1, 3), 17), (40, 4, (1,), 64),
                                              (33, 11, (1, 2, 3), 30), (12, 16, (1,), 9),
                                              (12, 17, (3,), 9), (20, 24, (1, 3), 5),
                                              (6, 32, (1,), 4), (6, 33, (1,), 4)])
def test_points(gpu_lib, nn, nm, comps, npts):
    p = _tower(nn, nm, 33, comps)
    rng = np.random.default_rng(npts)
    fi, fj = rng.uniform(-3.5, 3.5, (2, npts))
    fj[0] = -fi[0]                                      # f1 + f2 = 0
    if npts > 3:
        fi[1] = 0.0
        fj[2] = fi[2]
    bfm, brm = abi.bfm_points(p, fi, fj)
    want = O.msh_points(p, fi, fj)
    assert _rel(bfm, want) < 1e-12
    H1, H2, H3 = O.frf(p, fi), O.frf(p, fj), O.frf(p, fi + fj)
    fr = (H1[:, :, None, None] * H2[:, None, :, None] * np.conj(H3)[:, None, None, :]).real
    fr = fr.reshape(-1, nm ** 3, order="F").T
    assert _rel(brm, want * fr) < 1e-12
