"""The bootstraps around the ranges and batches of their kernels (needs an
MI355X), against the oracle on the same per-chunk results and draws."""
import numpy as np
import pytest

from lyspeq_amd import qml, synth
from lyspeq_amd.qml import QMLEngine
from oracle import bootstrap as ob

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def run():
    """An iterated engine with its spectra of two chunks: (engine, spectrum of
    each chunk, spectra, collapsed vectors, collapsed Fisher matrices)."""
    w = synth.desi_config(nchunks=16)
    eng = QMLEngine(w.binning, precision="fp64")
    synth.load_engine(eng, w)
    eng.commit()
    T = eng.T
    eng.iterate(np.zeros(T), np.zeros((T, T)), np.zeros((3, T)))
    infos, nch = eng.chunk_infos, len(eng.chunk_infos)
    res = [eng.chunk_result(c) for c in range(nch)]
    assert not any(r[2] for r in res) or all(r[2] for r in res)
    qso = (np.arange(nch) // 2).astype(np.int32)
    nqso = int(qso.max()) + 1
    of = [[c for c in range(nch) if qso[c] == s] for s in range(nqso)]
    key = lambda c: (infos[c].fisher_index_start, infos[c].n_q_matrices)
    col = [ob.collapse([(*key(c), res[c][1]) for c in cs]) for cs in of]
    fis = [ob.collapse_fisher([(*key(c), res[c][0]) for c in cs]) for cs in of]
    yield eng, qso, nqso, col, fis
    eng.close()


def _rel(a, b):
    return float(np.max(np.abs(a - b)) / np.max(np.abs(b)))


@pytest.mark.parametrize("nboots", [2, 15, 16, 31, 32, 33, 63, 64, 127, 128, 129, 1000])
def test_mean_and_covariance_ranges(run, nboots):
    """One range of realisations (under 32 for the covariance, under 128 for the
    mean) and several: the means and covariances of the engine's own
    realisations, at the tolerances of the other bootstrap tests."""
    print(f"[case] ranges of {nboots}", flush=True)
    eng, qso, nqso, col, _ = run
    R, mean, cov = eng.bootstrap(nboots, qso, nqso, seed=9)
    Ro = ob.realizations(qml.poisson_draws(9, nqso * nboots).reshape(nqso, nboots), col, eng.T)
    mo, co = ob.mean_covariance(R)
    assert _rel(R, Ro) < 1e-12 and _rel(mean, mo) < 1e-12 and _rel(cov, co) < 1e-11
    assert np.array_equal(cov, cov.T)


@pytest.mark.parametrize("nboots", [127, 128, 129, 160, 161, 256, 290])
def test_complete_bootstrap_batches(run, nboots):
    """Realisations are solved 128 at a time: full batches, a tail of one, tails
    around a group of 32, with an empty realisation (every weight zero) and one
    whose Fisher matrix is not positive definite in the first and in each later
    batch.  The bar is that of two Cholesky solves, 20 n cond eps."""
    print(f"[case] complete bootstrap of {nboots}", flush=True)
    eng, qso, nqso, col, fis = run
    rng = np.random.default_rng(nboots)
    W = rng.integers(1, 4, (nboots, nqso)).astype(np.int32)
    empty = [b for b in (5, 130, 260) if b < nboots]
    bad = [b for b in (40, 128, 200, 289) if b < nboots]
    W[empty] = 0
    W[bad, rng.integers(0, nqso, len(bad))] = -3
    X, valid, mean, cov = eng.bootstrap_complete(nboots, qso, nqso, weights=W)
    Xo, vo, systems = ob.complete_realizations(W, col, fis, eng.T, return_systems=True)
    assert np.array_equal(valid, vo) and X.shape == Xo.shape
    assert not valid[bad].any() and valid[empty].all() and valid.sum() == nboots - len(bad)
    at = np.cumsum(valid) - 1
    assert not X[at[empty]].any()
    eps = np.finfo(float).eps
    for xb, xo, (S, _) in zip(X, Xo, systems):
        d = np.sqrt(np.diag(S))
        scale = np.max(np.abs(xo * d))
        if scale > 0:
            assert np.max(np.abs((xb - xo) * d)) / scale < 20 * eng.T * np.linalg.cond(S / np.outer(d, d)) * eps
    mg, cg = ob.mean_covariance(X)
    assert _rel(mean, mg) < 1e-12 and _rel(cov, cg) < 1e-11
