"""The projection kernel at the edges of its launch shapes: node counts around its
tiles of 16 columns and its steps of 8 and 4 nodes, mode counts on both sides of every
template and of the chunks of 64, frequency lists that leave every remainder of a
group of 8, |f| = 0 with rho = 0, coherence above 1, results that underflow.

Modal force PSDs (bsahip_modal_psd_points) against numpy: sum over nodes of
A(n, i; f) Psi(p, i), A by its definition.  Tolerance 1e-12 of the largest entry: a sum
of at most 67^2 products, each factor correct to a few ulp, the argument |f| ln rho of
the power rounded once (|x| 2^-53 relative, 1e-14 where rho^|f| still counts)."""
import numpy as np
import pytest

from bsalib_amd import abi, synth
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _full(p, tc):
    m = np.zeros((p.nn, p.nn))
    iu = np.triu_indices(p.nn)
    m[iu] = p.nod_corr[:, tc - 1]
    return m + np.triu(m, 1).T


def _ref(p, f):
    psi = O.psi(p)
    out = np.zeros((p.nm, p.nm, f.size))
    for tc in p.tc:
        s = np.sqrt(O.eval_psd(p, f, int(tc)))
        rho, a = _full(p, int(tc)), psi[:, :, tc - 1]
        for q in range(f.size):
            with np.errstate(under="ignore"):
                co = rho ** abs(f[q])
            out[:, :, q] += ((a * s[q]) @ co * s[q]) @ a.T
    return out


def _check(p, f):
    r = abi.modal_psd_points(p, f)
    ref = _ref(p, f)
    assert np.abs(r - ref).max() < 1e-12 * np.abs(ref).max()


@pytest.mark.parametrize("nn", [1, 2, 3, 4, 5, 7, 8, 9, 12, 15, 16, 17, 31, 33, 67])
@pytest.mark.parametrize("nm", [1, 17])
def test_node_counts(gpu_lib, nn, nm):
    p = synth.tower(nn=nn, nm=nm, comps=(1, 3), natf=np.linspace(0.2, 3.0, nm), seed=nn)
    _check(p, np.array([0.0, 0.3, 1.7, -2.2, 40.0]))


@pytest.mark.parametrize("nm", [2, 16, 18, 32, 33, 48, 49, 64, 65, 130])
def test_mode_counts(gpu_lib, nm):
    p = synth.tower(nn=21, nm=nm, comps=(1, 2, 3), natf=np.linspace(0.2, 3.0, nm), seed=nm)
    _check(p, np.linspace(0.0, 3.0, 11))


@pytest.mark.parametrize("nf", [1, 7, 8, 9, 2047, 2051, 9001])
@pytest.mark.parametrize("nm", [3, 20, 40])
def test_frequency_groups(gpu_lib, nf, nm):
    p = synth.tower(nn=37, nm=nm, comps=(1,), natf=np.linspace(0.2, 3.0, nm), seed=nf)
    _check(p, np.linspace(0.01, 4.0, nf))


def test_limits_of_the_coherence(gpu_lib):
    p = synth.deck(nn=30, nm=4, comps=(1, 3), seed=2)
    rng = np.random.default_rng(0)
    rho = p.nod_corr.copy()
    at = rng.choice(rho.shape[0], 60, replace=False)
    rho[at[:20]] = 0.0                # uncorrelated pairs: rho^0 = 1, rho^|f| = 0
    rho[at[20:40]] = 1e-300           # underflows and subnormals
    rho[at[40:]] = 1.5                # grows with |f|
    p.nod_corr = rho
    _check(p, np.array([0.0, 0.5, 1.0, 1.05, 2.0, 3.9]))
    p.nod_corr[at[45], :] = -1.0      # no real power: NaN stays NaN
    assert np.isnan(abi.modal_psd_points(p, np.array([0.5]))).any()


@pytest.mark.parametrize("nm", [3, 20, 40, 60])
@pytest.mark.parametrize("bad", [-1.0, float("nan")])
def test_zero_frequency_with_no_real_power(gpu_lib, nm, bad):
    """rho < 0 or NaN: rho^0 is 1 all the same, in every place of a group of frequencies
    and in both table layouts; every other power is NaN."""
    p = synth.tower(nn=13, nm=nm, comps=(1, 3), natf=np.linspace(0.2, 3.0, nm), seed=5)
    one = synth.tower(nn=13, nm=nm, comps=(1, 3), natf=np.linspace(0.2, 3.0, nm), seed=5)
    at = [3, 20, 77]                       # pairs of different nodes
    p.nod_corr, one.nod_corr = p.nod_corr.copy(), one.nod_corr.copy()
    p.nod_corr[at], one.nod_corr[at] = bad, 1.0
    for f in (np.zeros(1), np.array([0.5, 0.0, 1.0, 0.0, 0.0, 2.0, 0.25, 3.0, 0.0])):
        r, ref = abi.modal_psd_points(p, f), _ref(one, f)
        z = f == 0.0
        assert np.isnan(r[:, :, ~z]).all()
        assert np.abs(r[:, :, z] - ref[:, :, z]).max() < 1e-12 * np.abs(ref[:, :, z]).max()
    if nm <= 32:
        bfm, _ = abi.bfm_points(p, np.zeros(2), np.zeros(2))
        want = O.msh_points(one, np.zeros(2), np.zeros(2))
        assert np.abs(bfm - want).max() < 1e-12 * np.abs(want).max()


@pytest.mark.parametrize("psd_id", [1, 2, 3, 5])
def test_frequencies_that_are_not_finite(gpu_lib, psd_id):
    """NaN and infinite frequencies give NaN and leave their neighbours alone."""
    p = synth.tower(nn=9, nm=3, comps=(1, 3), natf=np.linspace(0.2, 3.0, 3), seed=5)
    b = abi.Bound(p, psd_id=psd_id)
    f = np.array([0.0, np.nan, 1.0, np.inf, 2.0, -np.inf, 0.5, 3.0, np.nan])
    ok = np.isfinite(f)
    r = abi.modal_psd_points(p, f, bound=b)
    assert np.isnan(r[:, :, ~ok]).all()
    assert np.array_equal(r[:, :, ok], abi.modal_psd_points(p, f[ok], bound=b))
