"""Modal PSD moments and batch table launches at the edges of their shapes: frequency
counts around the blocks of 64, mode counts around the tiles of 16 and chunks of 32,
contraction lengths that need padding; a batch that mixes them must give each
structure's own run in every mode.

Second moments against numpy (oracle.modal_psd), tolerance 1e-12 of the largest entry:
sums of at most 3 * 40 * 257 products, each factor correct to a few ulp."""
import numpy as np
import pytest

from bsalib_amd import abi, synth
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _tower(nn, nm, nfh, comps=(1, 3)):
    return synth.tower(nn=nn, nm=nm, comps=comps, natf=np.linspace(0.2, 3.0, nm), nfreqs=nfh,
                       df=4.0 / nfh, seed=nn + nm + nfh)


def _rel(a, b):
    return np.abs(a - b).max() / np.abs(b).max()


@pytest.mark.parametrize("nn,nm,nfh,comps", [(1, 1, 2, (1,)), (3, 1, 63, (1,)), (9, 2, 64, (1, 3)),
                                             (40, 15, 65, (1, 2, 3)), (17, 16, 128, (1,)),
                                             (23, 17, 129, (3,)), (12, 33, 257, (1, 3)),
                                             (5, 70, 33, (1,))])
def test_second_moments(gpu_lib, nn, nm, nfh, comps):
    p = _tower(nn, nm, nfh, comps)
    m = O.modal_psd(p)
    for kw in ({}, {"deterministic": True}, {"exact": True}):
        r = abi.classic_run(p, bisp=False, **kw)
        for k in ("m2mf", "m2mr"):
            assert _rel(r[k], m[k]) < 1e-12, (k, kw)
    a = abi.classic_run(p, bisp=False)
    d = abi.classic_run(p, bisp=False, deterministic=True)
    assert _rel(a["m2o2mr"], d["m2o2mr"]) < 1e-13


@pytest.mark.parametrize("prec", ["fp64", "fp32", "bf16x3"])
def test_mixed_batch(gpu_lib, prec):
    probs = [_tower(7, 2, 17), _tower(33, 17, 40), _tower(20, 5, 65, (1,)), _tower(1, 1, 3, (1,)),
             _tower(21, 36, 9), _tower(50, 3, 33, (1, 2, 3))]
    b = abi.Batch(probs, prec=prec)
    want = [abi.Plan(p, prec=prec).run() for p in probs]
    for mode in (2, 0, 1, 0, 2):
        r = b.run(mode=mode)
        for i, w in enumerate(want):
            for k in ("m3mf", "m3mr", "m2mr"):
                # atomic sums: the order of the terms varies
                assert _rel(r[k][i], w[k]) < 1e-12, (mode, i, k)
    b.close()
