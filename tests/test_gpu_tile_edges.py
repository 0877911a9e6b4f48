"""The chunk step at the edges of its kernels' tiles (needs an MI355X): pixel
counts around the 16-column panels, the 64-blocks and the 128-tiles, FP64
against the oracle at the parity bar."""
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
