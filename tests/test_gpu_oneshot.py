"""One-shot calls share scratch and staging memory: calls of growing and shrinking
sizes through different entry points, in any order, from several threads and after a
refused call, give what each gives by itself; results above the staged size and inputs
above the staged part size too.  Ordered sums make equal calls equal bit for bit."""
import ctypes as C
import resource
import threading

import numpy as np
import pytest

from bsalib_amd import abi, synth
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _tower(nn, nm, nfh, comps=(1, 3)):
    return synth.tower(nn=nn, nm=nm, comps=comps, natf=np.linspace(0.2, 3.0, nm), nfreqs=nfh,
                       df=4.0 / nfh, seed=nn + nm)


def _calls():
    """One-shot calls; 42 modes and 530 nodes pass the staged sizes, 300 nodes with 513
    frequencies the scratch that is kept."""
    big, mid, small, many = _tower(530, 3, 9), _tower(120, 17, 40), _tower(7, 2, 17), _tower(30, 42, 5)
    wide = _tower(300, 15, 513, (1, 2, 3))
    pts = np.linspace(-3.0, 3.0, 23), np.linspace(2.5, -1.5, 23)

    def run(p, **kw):
        return lambda: {k: v for k, v in abi.classic_run(p, deterministic=True, **kw).items()}

    return [run(mid), run(small), run(big), run(many), run(small, exact=True), run(mid, bisp=False),
            run(mid, psd=False, prec="bf16x3"), run(wide, bisp=False, prec="bf16x3"),
            lambda: abi.classic_bispectra_sel(small, [1, 8]),
            lambda: abi.classic_bispectra_sel(mid, [5], exact=True),
            lambda: abi.classic_bispectra_sel(mid, [5], only_diag=True),
            lambda: dict(zip("fr", abi.bfm_points(mid, *pts))),
            lambda: dict(zip("fr", abi.bfm_points(small, *pts, only_diag=True)))]


def _same(a, b):
    return all(np.array_equal(a[k], b[k]) for k in a)


def test_order_and_threads(gpu_lib):
    calls = _calls()
    want = [c() for c in calls]
    rng = np.random.default_rng(1)
    for i in np.concatenate([rng.permutation(len(calls)) for _ in range(3)]):
        if i % 4 == 0:
            with pytest.raises(abi.BsaHipError):
                abi.classic_bispectra_sel(_tower(7, 2, 17), [0])
        assert _same(want[i], calls[i]()), i
    bad = []

    def work(seed):
        for i in np.random.default_rng(seed).permutation(len(calls)):
            if not _same(want[i], calls[i]()):
                bad.append(i)

    ts = [threading.Thread(target=work, args=(s,)) for s in (2, 3, 4)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad


def test_second_moments_above_the_staged_sizes(gpu_lib):
    """Tolerance 1e-12 of the largest entry, sums of at most 2 * 530 * 17 products."""
    for p in (_tower(530, 3, 9), _tower(30, 42, 5)):
        o = O.modal_psd(p)
        r = abi.classic_run(p)
        for k in ("m2mf", "m2mr", "m2o2mr"):
            assert np.abs(r[k] - o[k]).max() < 1e-12 * np.abs(o[k]).max()


def test_refused_diagonal_grid(gpu_lib):
    """A diagonal run whose plane is too large for one launch is refused before anything
    starts on the side stream; the calls after it have the scratch to themselves."""
    p = _tower(9, 4, 33)
    o = O.classic_diag(p)
    want = abi.classic_run(p, only_diag=True)
    huge = _tower(1, 256, 33100, (1,))
    for _ in range(3):
        with pytest.raises(abi.BsaHipError, match="too large"):
            abi.classic_run(huge, only_diag=True)
        r = abi.classic_run(p, only_diag=True)
        for k in ("m2mf", "m2mr", "m3mf", "m3mr"):
            assert np.abs(r[k] - want[k]).max() <= 1e-14 * np.abs(want[k]).max()
            assert np.abs(r[k] - o[k]).max() < 1e-12 * np.abs(o[k]).max()


def test_pinned_coherence_table(gpu_lib, tmp_path):
    """A coherence table in pinned memory, larger than the staged parts, is read when the
    call returns, also by the calls that do not wait for their results (a Mesher loaded
    from its checkpoint): the caller may overwrite it."""
    def deck():
        return synth.tower(nn=800, nm=2, comps=(1, 2), natf=np.array([0.3, 0.8]),
                           xi=np.array([0.02, 0.03]), nfreqs=9, df=0.5, seed=3)

    kw = dict(bkg_base_rfmnt=4, tile_cells=2, bkg_peakw=2.0)
    m = abi.Mesher(deck(), **kw)
    want = m.run(levels=2)
    m.save(tmp_path / "zones")
    m.close()
    p = deck()
    table = p.nod_corr
    at = C.c_void_p()                   # of the HIP runtime that the library is linked to
    assert gpu_lib.lib().hipHostMalloc(C.byref(at), C.c_size_t(8 * table.size), C.c_uint(0)) == 0
    pinned = np.ctypeslib.as_array(C.cast(at, C.POINTER(C.c_double)), (table.size,))
    for _ in range(3):
        p.nod_corr = pinned.reshape(table.shape, order="F")
        p.nod_corr[:] = table
        b = abi.Bound(p)
        assert np.shares_memory(b.keep["nod_corr"], pinned)
        m = abi.Mesher(p, bound=b, load=tmp_path / "zones", **kw)
        pinned[::-1] = 0.5
        r = m.run(levels=2)
        m.close()
        for k in ("m3mf", "m3mr"):
            assert np.abs(r[k] - want[k]).max() <= 1e-12 * np.abs(want[k]).max()
    del b, p
    assert gpu_lib.lib().hipHostFree(at) == 0


def test_refused_grids_make_no_tables(gpu_lib):
    """A grid that no launch can hold is refused before a list of its frequencies (2 GB
    and more here) is made or sent: the process does not grow, and an allocation that
    fails cannot leave the C entry by an exception."""
    p = _tower(3, 1, 9, (1,))
    p.nfreqs = 1 << 28
    before = resource.getrusage(resource.RUSAGE_SELF).ru_maxrss
    for make in (lambda: abi.classic_run(p), lambda: abi.classic_run(p, exact=True, prec="bf16x3"),
                 lambda: abi.classic_run(p, only_diag=True), lambda: abi.Plan(p, prec="fp32"),
                 lambda: abi.Batch([p])):
        with pytest.raises(abi.BsaHipError, match="too large"):
            make()
    p.nfreqs = 2 ** 31 - 1                               # the list would hold 2^32 - 3
    for kw in ({"exact": True}, {}, {"only_diag": True}):
        with pytest.raises(abi.BsaHipError, match="too large"):
            abi.classic_run(p, **kw)
    assert resource.getrusage(resource.RUSAGE_SELF).ru_maxrss - before < 256 << 10


def _free():
    a, b = C.c_size_t(0), C.c_size_t(0)
    assert abi.lib().hipMemGetInfo(C.byref(a), C.byref(b)) == 0
    return a.value


def test_scratch_of_other_calls_is_kept(gpu_lib):
    """A small moments run keeps the scratch of a large call of another kind (a third of a
    gigabyte, more than plans keep), and a large moments run gives its own back."""
    small, wide, sel = _tower(7, 2, 17), _tower(300, 15, 513, (1, 2, 3)), _tower(7, 3, 513)
    abi.classic_run(small)
    abi.classic_bispectra_sel(sel, np.arange(1, 21))
    before = _free()
    abi.classic_run(small)
    assert abs(_free() - before) < 32 << 20
    abi.classic_run(wide, bisp=False, prec="bf16x3")            # 500 MB of tables
    assert abs(_free() - before) < 288 << 20
    abi.classic_run(small)
    assert abs(_free() - before) < 288 << 20


def test_scratch_of_few_frequencies(gpu_lib):
    """The diagonal bispectra of two frequencies take tables of two columns, not of whole
    tiles: 60 modes, 900 nodes, 3 components 2.6 MB, where 128 columns take 167."""
    p = _tower(900, 60, 2, (1, 2, 3))
    want = abi.classic_bispectra_sel(p, [1, 60], only_diag=True)
    abi.lib().bsahip_finalise()
    abi.init(0)
    before = _free()
    r = abi.classic_bispectra_sel(p, [1, 60], only_diag=True)
    assert before - _free() < 64 << 20
    for k in ("bisp_f", "bisp_r"):
        assert np.array_equal(r[k], want[k])
