"""The atomic sums of the FP64 third moments lose next to nothing to the order of their
additions: the moments equal the fixed-order compensated sums of the same contributions,
for all wave tiles, with few copies of the moments and many, and in batches.

Tolerance 4 * 2^-53 of the largest entry: a copy takes about four additions, so that its
sum is off by at most four roundings of 2^-53 of its largest partial sum, and the copies'
own sum and the fixed-order one are compensated."""
import numpy as np
import pytest

from bsalib_amd import abi, synth

pytestmark = pytest.mark.gpu
TOL = 4 * 2.0 ** -53


def _deck(nn, nm, nfh, seed):
    return synth.deck(nn=nn, nm=nm, comps=(1, 3), nfreqs=nfh, df=4.0 / (nfh - 1), seed=seed,
                      u10=22.0 + seed, span=10.0 * (10.0 * nn) ** 0.5)


def _off(a, b):
    return max(np.abs(a[k] - b[k]).max() / np.abs(b[k]).max() for k in ("m3mf", "m3mr"))


@pytest.mark.parametrize("nn,nm,nfh", [(20, 1, 48), (20, 3, 65), (40, 9, 101), (40, 14, 60),
                                       (30, 2, 1025), (60, 16, 257)])
def test_as_ordered_sums(gpu_lib, nn, nm, nfh):
    for seed in range(6):
        p = _deck(nn, nm, nfh, seed)
        want = abi.classic_run(p, psd=False, deterministic=True)
        plan = abi.Plan(p)
        for r in (abi.classic_run(p), plan.run(), plan.run()):
            assert _off(r, want) <= TOL, seed
        plan.close()


def test_batches(gpu_lib):
    """Structures whose own launch takes the batch's tile: the same contributions."""
    probs = [_deck(20 + s, 3, 65 + s, s) for s in range(12)] + [_deck(20, 6, 90, 3), _deck(9, 2, 20, 3)]
    b = abi.Batch(probs)
    want = [abi.classic_run(p, psd=False, deterministic=True) for p in probs]
    for mode in (0, 2, 1, 0, 0):
        r = b.run(mode=mode)
        for i, w in enumerate(want[:-1]):
            assert _off({k: r[k][i] for k in ("m3mf", "m3mr")}, w) <= TOL, (mode, i)
        assert _off({k: r[k][-1] for k in ("m3mf", "m3mr")}, want[-1]) < 1e-13
    b.close()
