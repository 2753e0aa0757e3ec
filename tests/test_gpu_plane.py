"""The G contraction with its plane quadrature at the edges of its tiles and of its
epilogue classes: half grids around 16 and 64 points, modes that share a block of 16
rows, one mode, contractions from one padded chunk on, against
oracle.classic_factorised, for every quadrature rule, the plane continued beyond
+-fmax and the generic epilogue.

Tolerances, of the largest entry: FP64 1e-12 (sums of at most 3 * 60 * 257^2 terms in
blocks, each factor correct to a few ulp); FP32 and BF16x3 1e-5 (24 mantissa bits of the
operands or products dropped below 2^-16 of them, and FP32 sums of at most 180 terms)."""
import numpy as np
import pytest

from bsalib_amd import abi, synth
from oracle import oracle as O

pytestmark = pytest.mark.gpu

SIZES = [(1, 1, 2, (1,)), (7, 1, 129, (1,)), (5, 2, 15, (1, 3)), (9, 3, 16, (1,)), (20, 5, 17, (3,)),
         (33, 4, 63, (1, 3)), (16, 3, 64, (1,)), (60, 7, 65, (1, 2, 3)), (24, 17, 9, (1, 3)),
         (32, 12, 47, (1,)), (45, 19, 33, (1, 3)), (60, 24, 41, (1,))]


def _rel(a, b):
    return np.abs(a - b).max() / np.abs(b).max()


@pytest.mark.parametrize("nn,nm,nfh,comps", SIZES)
def test_third_moments(gpu_lib, nn, nm, nfh, comps):
    p = synth.tower(nn=nn, nm=nm, comps=comps, natf=np.linspace(0.2, 3.0, nm), nfreqs=nfh,
                    df=4.0 / nfh, seed=nn + nm + nfh)
    for rule, exact in (("vect", False), ("riemann", False), ("trapezoid", False), ("vect", True)):
        o = O.classic_factorised(p, rule=rule, truncate=not exact)
        for prec, tol in (("fp64", 1e-12), ("fp32", 1e-5), ("bf16x3", 1e-5)):
            for gen in (False, True):
                r = abi.classic_run(p, quad=rule, prec=prec, psd=False, exact=exact, epi_generic=gen)
                for k in ("m3mf", "m3mr"):
                    assert _rel(r[k], o[k]) < tol, (k, rule, exact, prec, gen)


@pytest.mark.parametrize("nn,nm,nfh", [(40, 30, 60), (10, 8, 100), (100, 40, 70)])
def test_tiles_agree(gpu_lib, nn, nm, nfh):
    """Launches that take the smaller and the larger wave tiles: the same moments as the
    generic epilogue and as ordered sums give, to the order of the terms."""
    p = synth.tower(nn=nn, nm=nm, comps=(1, 3), natf=np.linspace(0.2, 3.0, nm), nfreqs=nfh,
                    df=4.0 / nfh, seed=nm)
    a = abi.classic_run(p, psd=False)
    for kw in ({"epi_generic": True}, {"deterministic": True}):
        b = abi.classic_run(p, psd=False, **kw)
        for k in ("m3mf", "m3mr"):
            assert _rel(a[k], b[k]) < 1e-12, (k, kw)
