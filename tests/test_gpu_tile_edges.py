"""The chunk step at the edges of its kernels' tiles (needs an MI355X): pixel
counts around the 16-column panels, the 64-blocks and the 128-tiles, FP64
against the oracle at the parity bar; and member counts around the 16-blocks of
the split Gram, against the FP64 engine at the split products' parity bar."""
import numpy as np
import pytest

import parity as P
from lyspeq_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes", [(17, 33, 63), (64, 65, 80, 127), (128, 129, 192, 256)])
def test_pixel_counts_at_tile_edges(sizes):
    print(f"[case] N = {sizes}", flush=True)
    w = synth.cpu_reference_config(nchunks=len(sizes))
    w.binning.max_forest_length_v = 1.0e3
    for c, n in zip(w.chunks, sizes):
        for k in ("wave", "delta", "ivar"):
            c[k] = c[k][:n].copy()
        c["ivar"][0] = c["ivar"][0] or 10.0
        c["ivar"][n - 1] = c["ivar"][n - 1] or 10.0
    th = P.theta_perturbed(w.binning, w.pd13, 0.05, 61)
    idx = range(len(sizes))
    oout, oF, od = P.run_oracle(w, th, idx)
    assert len(oout) == len(sizes)
    eng, out, F, dbt = P.run_engine(w, th, idx, precision="fp64")
    eng.close()
    floor, xout, _ = P.oracle_floor(w, th, idx, oout)
    P.assert_chunks_fp64(out, oout, f"N {sizes}", floor=floor, exact=xout)


@pytest.mark.parametrize("members", [16, 17, 33, 50, 62])
@pytest.mark.parametrize("precision", ["bf16x3", "bf16x4"])
def test_member_counts_at_gram_blocks(members, precision):
    print(f"[case] m = {members} {precision}", flush=True)
    w = synth.cpu_reference_config(nchunks=2, with_tables=False)
    b = w.binning
    b.max_forest_length_v = 1.0e3
    b.nklog, b.nklin = 0, members - 2          # one z bin: members = bands + 2
    b.dklin = 0.04 / b.nklin
    for c in w.chunks:
        for k in ("wave", "delta", "ivar"):
            c[k] = c[k][:100].copy()
    w = synth._finish_tables(w, True)
    th = np.full(b.nklin, 0.1)
    F = {}
    for p in ("fp64", precision):
        eng, out, F[p], _ = P.run_engine(w, th, range(2), precision=p)
        eng.close()
        assert all(o[2] for o in out.values())
    err = P.fisher_norm_err(F[precision], F["fp64"])
    print(f"[err] {err:.2e}", flush=True)
    assert err < P.MIXED_TOL[("desi", "bf16x3")]["F_norm"]
