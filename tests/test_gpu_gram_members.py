"""The Gram matrix at member counts around its blocks (needs an MI355X): the
split products' kernel for up to 128 members holds one row block a wave up to
64 and two above, over 128 the tiled one takes over.  FP64 against the oracle at
the parity bar; the split products bit for bit against their other kernel, and
against FP64 at their parity bar."""
import numpy as np
import pytest

import parity as P
from lyspeq_amd import synth
from lyspeq_amd.qml import QMLEngine

pytestmark = pytest.mark.gpu

# z bins that a chunk of 100 pixels at z = 2.4 spans: (first centre, width)
ZBINS = {1: (2.4, 0.2), 2: (2.3, 0.2), 3: (2.36, 0.04), 5: (2.362, 0.018)}


def _workload(members, nzq, nk):
    w = synth.cpu_reference_config(nchunks=2, with_tables=False)
    b = w.binning
    b.max_forest_length_v = 1.0e3
    b.nklog, b.nklin, b.dklin = 0, nk, 0.04 / nk
    b.nz, (b.z0, b.z_bin_width) = nzq, ZBINS[nzq]
    for c in w.chunks:
        for k in ("wave", "delta", "ivar"):
            c[k] = c[k][78:178].copy()
        c["ivar"][0] = c["ivar"][0] or 10.0
        c["ivar"][-1] = c["ivar"][-1] or 10.0
    assert nzq * nk + 2 == members
    return synth._finish_tables(w, True)


def _run(w, precision, gram=None):
    eng = QMLEngine(w.binning, precision=precision)
    got = synth.load_engine(eng, w)
    if gram:
        eng.set_kernel_stages(3, 3, gram)
    eng.commit()
    T = eng.T
    F, dbt = np.zeros((T, T)), np.zeros((3, T))
    eng.iterate(np.full(T, 0.1), F, dbt)
    m = max(i.n_stored for i in eng.chunk_infos) + 2
    eng.close()
    return len(got), m, F, dbt


@pytest.mark.parametrize("members,nzq,nk", [(63, 1, 61), (64, 2, 31), (65, 3, 21), (66, 2, 32), (80, 3, 26), (82, 2, 40),
                                            (96, 2, 47), (97, 5, 19), (112, 2, 55), (113, 3, 37), (127, 5, 25),
                                            (128, 2, 63), (131, 3, 43), (192, 5, 38)])
def test_member_counts(members, nzq, nk):
    print(f"[case] gram members {members}", flush=True)
    w = _workload(members, nzq, nk)
    n, m, F64, d64 = _run(w, "fp64")
    assert (n, m) == (2, members)
    oout, oF, od = P.run_oracle(w, np.full(nzq * nk, 0.1), range(2))
    P.assert_fp64(F64, d64, oF, od, f"gram members {members}")
    for precision in ("bf16x3", "bf16x4"):
        ref = _run(w, precision, gram=1)[2]
        got = _run(w, precision, gram=3)[2]
        assert np.array_equal(got, ref), precision
        assert P.fisher_norm_err(got, F64) < P.MIXED_TOL[("desi", "bf16x3")]["F_norm"]
