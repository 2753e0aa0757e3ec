"""The ONLY_DIAG moments at the edges of their launch shapes: half grids around the
tiles of 64, short and long contractions, mode counts around 16 and 32, against
oracle.classic_diag, with the classes of the plane quadrature and the generic one.

Tolerance 1e-12 of the largest entry: sums of at most 3 * 700 * 257^2 terms in blocks,
each factor correct to a few ulp."""
import numpy as np
import pytest

from bsalib_amd import abi, synth
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return np.abs(a - b).max() / np.abs(b).max()


@pytest.mark.parametrize("nn,nm,nfh,comps", [(1, 1, 2, (1,)), (5, 2, 63, (1, 3)), (11, 3, 64, (1,)),
                                             (300, 4, 65, (1, 3)), (700, 2, 66, (1,)),
                                             (33, 16, 20, (1, 2, 3)), (20, 17, 33, (3,)),
                                             (9, 35, 17, (1,)), (170, 2, 129, (1, 2, 3))])
def test_moments(gpu_lib, nn, nm, nfh, comps):
    p = synth.tower(nn=nn, nm=nm, comps=comps, natf=np.linspace(0.2, 3.0, nm), nfreqs=nfh,
                    df=4.0 / nfh, seed=nn)
    o = O.classic_diag(p)
    for kw in ({}, {"epi_generic": True}):
        r = abi.classic_run(p, only_diag=True, **kw)
        for k in ("m2mf", "m2mr", "m3mf", "m3mr"):
            assert _rel(r[k], o[k]) < 1e-12, (k, kw)
    only2 = abi.classic_run(p, only_diag=True, bisp=False)
    only3 = abi.classic_run(p, only_diag=True, psd=False)
    assert _rel(only2["m2mr"], o["m2mr"]) < 1e-12 and not only2["m3mr"].any()
    assert _rel(only3["m3mr"], o["m3mr"]) < 1e-12 and not only3["m2mr"].any()
