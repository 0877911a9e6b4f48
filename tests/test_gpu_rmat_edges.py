"""Q_k with a resolution matrix at the edges of its kernels (needs an MI355X).

The quadrature in k and the band-edge form, against the oracle's
extended-precision run: chunks just below, at and above whole 64-pixel tiles,
each row shape of R, bands of few and of many nodes, and one too wide for the
quadrature.  The bar is that of the rounding of v itself (about c eps = 3e-11
km/s) through the phase k v, k < 0.1 s/km, with a factor of three.
"""
import numpy as np
import pytest

import parity as P
from lyspeq_amd import qml, synth
from lyspeq_amd.qml import QMLEngine
from oracle.chunk import Chunk as OracleChunk

pytestmark = pytest.mark.gpu
TOL = 1e-11


def _bins(nklin, dklin):
    return qml.Binning(k0=0.0, nklin=nklin, dklin=dklin, nklog=3, dklog=0.2, z0=2.0, z_bin_width=0.2, nz=13, method=1,
                       cont_logl_order=1, cont_lam_order=-1, max_forest_length_v=3.0e3)


@pytest.mark.parametrize("n", [64, 65, 127, 128, 129, 320])
@pytest.mark.parametrize("kind,bins", [("dia", (6, 0.001)), ("oversampled", (6, 0.004)), ("oversampled", (1, 0.09)),
                                       ("dia", (1, 0.09))])
def test_band_matrices(kind, bins, n):
    print(f"[case] rmat bands {kind} {bins} {n}", flush=True)
    w = synth.rmat_config(seed=11, nchunks=1, n_range=(n, n), kind=kind, with_tables=False)
    w.binning = _bins(*bins)
    b = P.oracle_bins(w.binning)
    w.deriv = synth.derivative_tables(w.binning.kband_edges(), w.pairs, w.nv, w.v_length)
    w.signal = synth.signal_tables(w.binning, w.pairs, w.nv, w.v_length, w.nz_table, w.pd13)
    c = w.chunks[0]
    assert c["wave"].size == n
    ch = OracleChunk(b, P.oracle_tables(w), c["wave"], c["delta"], c["ivar"], c["R"], rmat=P.oracle_rmat(c), exact=True)
    v, _ = ch.vz_matrices()
    eng = QMLEngine(w.binning, precision="fp64")
    try:
        (_, cid), = synth.load_engine(eng, w)
        eng.commit()
        for i_kz in list(ch.stored)[:ch.kbin_upp]:
            kn = (i_kz + ch.fisher_index_start) % b.nk
            want, got = ch.q_base(v, kn), eng.chunk_matrix(cid, qml.CMAT_Q, i_kz)
            assert np.array_equal(got, got.T)
            err = float(np.max(np.abs(got - want)) / np.max(np.abs(want)))
            print(f"[err] band {kn}: {err:.2e}", flush=True)
            assert err < TOL
    finally:
        eng.close()
