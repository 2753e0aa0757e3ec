"""Point lists on a card that is nearly full: the point kernel's table has 16 or 32 columns
for any count of modes, and where it finds no memory the general kernel takes the call with
its own of as many columns as modes.  The rest of the card is held by one allocation that
no kernel touches.

Against the same calls with the card free, 1e-12 of the largest entry: sums of at most
3 * 400 products, another order of the terms in the general kernel."""
import contextlib
import ctypes as C

import numpy as np
import pytest

from bsalib_amd import abi, synth

pytestmark = pytest.mark.gpu


def _free(L):
    a, b = C.c_size_t(0), C.c_size_t(0)
    assert L.hipMemGetInfo(C.byref(a), C.byref(b)) == 0
    return a.value


@contextlib.contextmanager
def _card_with(L, left):
    """The card with `left` bytes free."""
    at = C.c_void_p()
    assert L.hipMalloc(C.byref(at), C.c_size_t(_free(L) - left)) == 0
    try:
        yield
    finally:
        assert L.hipFree(at) == 0


def _same(a, b):
    return np.abs(a - b).max() <= 1e-12 * np.abs(b).max()


def test_points(gpu_lib):
    """21600 points, one mode, 400 nodes: 3.4 GB of table (some 64800 frequencies), 1.2 GB
    free; the general kernel's takes 0.2 GB."""
    L = gpu_lib.lib()
    p = synth.tower(nn=400, nm=1, comps=(1,), natf=np.array([0.2]), nfreqs=9, df=0.5, seed=1)
    b = abi.Bound(p)
    rng = np.random.default_rng(0)
    few, many = rng.uniform(-3, 3, (2, 50)), rng.uniform(-3, 3, (2, 21600))
    many[:, :50] = few
    want = abi.bfm_points(p, *few, bound=b)
    L.bsahip_finalise()                              # gives back what earlier calls left
    abi.init(0)
    with _card_with(L, 1200 << 20):
        r = abi.bfm_points(p, *many, bound=b)
        again = abi.bfm_points(p, *few, bound=b)
    for k in range(2):
        assert np.isfinite(r[k]).all() and _same(r[k][:, :50], want[k]) and _same(again[k], want[k])
