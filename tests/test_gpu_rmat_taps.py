"""Resolution matrices of the fewest and the most taps a row (needs an MI355X)."""
import numpy as np
import pytest

import parity as P
from lyspeq_amd import qml, synth
from lyspeq_amd.qml import QMLEngine
from oracle.chunk import Chunk as OracleChunk

pytestmark = pytest.mark.gpu


def _bins(nklin, dklin):
    return qml.Binning(k0=0.0, nklin=nklin, dklin=dklin, nklog=3, dklog=0.2, z0=2.0, z_bin_width=0.2, nz=13, method=1,
                       cont_logl_order=1, cont_lam_order=-1, max_forest_length_v=3.0e3)


def _workload(bins, n, shapes, seed=21):
    """One chunk of n pixels per (kind, oversampling, nelem)."""
    w = synth.rmat_config(seed=seed, nchunks=len(shapes), n_range=(n, n), kind="dia", with_tables=False)
    w.binning = _bins(*bins)
    assert len(w.chunks) == len(shapes)
    for c, (kind, over, nelem) in zip(w.chunks, shapes):
        sigma = c["wave"] / (c["R"] * synth.ONE_SIGMA_2_FWHM)
        vals = synth._gaussian_rows(c["wave"], sigma, nelem, over)
        if kind == "oversampled" and over == 1:      # the rows of the diagonal form's matrix
            h, rows = nelem // 2, np.zeros((n, nelem))
            for t in range(nelem):
                i = np.arange(max(0, h - t), min(n, n + h - t))
                rows[i, t] = vals[nelem - 1 - t, i + t - h]
            vals = rows
        c["rmat"] = dict(kind=kind, nelem=nelem, oversampling=over, values=vals)
    w.deriv = synth.derivative_tables(w.binning.kband_edges(), w.pairs, w.nv, w.v_length)
    w.signal = synth.signal_tables(w.binning, w.pairs, w.nv, w.v_length, w.nz_table, w.pd13)
    return w


def _oracle(w, c):
    return OracleChunk(P.oracle_bins(w.binning), P.oracle_tables(w), c["wave"], c["delta"], c["ivar"], c["R"],
                       rmat=P.oracle_rmat(c), exact=True)


# bands of a few nodes, and one too wide for the quadrature, by its edges
@pytest.mark.parametrize("bins", [(6, 0.002), (1, 0.09)])
@pytest.mark.parametrize("n", [65, 320, 321, 328, 329])
@pytest.mark.parametrize("shape", [("dia", 1, 1), ("dia", 1, 3), ("oversampled", 1, 1), ("oversampled", 1, 5)])
def test_band_matrices_of_few_taps(bins, n, shape):
    """The last grid point is a pixel's own where a row has one tap or the
    grid is not oversampled.  The bar is the rounding of the phase k v."""
    print(f"[case] few taps {shape} {bins} {n}", flush=True)
    w = _workload(bins, n, [shape])
    ch = _oracle(w, w.chunks[0])
    v, _ = ch.vz_matrices()
    eng = QMLEngine(w.binning, precision="fp64")
    try:
        (_, cid), = synth.load_engine(eng, w)
        eng.commit()
        for i_kz in list(ch.stored)[:ch.kbin_upp]:
            kn = (i_kz + ch.fisher_index_start) % w.binning.nk
            want, got = ch.q_base(v, kn), eng.chunk_matrix(cid, qml.CMAT_Q, i_kz)
            assert np.max(np.abs(got - want)) < 1e-11 * np.max(np.abs(want)), kn
    finally:
        eng.close()


LONG = [("dia", 1, 11), ("dia", 1, 57), ("dia", 1, 59), ("dia", 1, 81), ("oversampled", 2, 65), ("oversampled", 3, 51),
        ("oversampled", 5, 21)]


@pytest.mark.parametrize("n", [64, 130])
def test_signal_of_long_rows(n):
    """R rows up to the most taps that are taken, in one batch: S against the
    oracle's extended-precision run (the bar of the rounding of v), and each
    chunk's S, F and d, b, t the same, bit for bit, alone and with the others."""
    print(f"[case] long rows {n}", flush=True)
    w = _workload((6, 0.004), n, LONG)
    T = w.binning.total_kz_bins

    def run(chunks):
        eng = QMLEngine(w.binning, precision="fp64")
        got = synth.load_engine(eng, w, chunks)
        eng.commit()
        eng.iterate(np.full(T, 0.1), np.zeros((T, T)), np.zeros((3, T)))
        res = {i: (*eng.chunk_result(cid)[:2], eng.chunk_matrix(cid, qml.CMAT_SFID)) for i, cid in got}
        eng.close()
        return res

    together = run(list(range(len(LONG))))
    assert len(together) == len(LONG)
    for i, c in enumerate(w.chunks):
        ch = _oracle(w, c)
        want, got = ch.signal_matrix(*ch.vz_matrices()), together[i][2]
        assert np.array_equal(got, got.T)
        assert np.max(np.abs(got - want)) < 1e-11 * np.max(np.abs(want)), LONG[i]
        for a, b in zip(together[i], run([i])[i]):
            assert np.array_equal(a, b), LONG[i]
