"""The bootstrap's kernels at the edges of their ranges (needs an MI355X)."""
import numpy as np
import pytest

from lyspeq_amd import synth
from lyspeq_amd.qml import QMLEngine
from oracle import bootstrap as ob

pytestmark = pytest.mark.gpu


# counts around what one workgroup ranks at once (1024), holds in LDS (3072)
# and samples (512); distributions with ties, one value, both signs, infinities
@pytest.mark.parametrize("nboots", [1, 2, 255, 512, 1023, 1024, 1025, 1501, 3072, 3073, 3074, 6000, 6001])
def test_median_selection_edges(nboots):
    print(f"[case] median of {nboots}", flush=True)
    rng = np.random.default_rng(nboots)
    R = rng.standard_normal((nboots, 6))
    R[:, 1] = np.round(R[:, 1], 1)                      # ties
    R[:, 2] = 3.25                                      # one value
    R[:, 3] = np.exp(8 * R[:, 3])                       # many decades
    R[:, 4] = np.where(R[:, 4] > 0.8, np.inf, R[:, 4])  # beyond the median's rank
    R[:, 5] = np.sort(R[:, 5])                          # an order the sample follows
    if nboots <= 2:
        R[:, 4] = 1.0
    eng = QMLEngine(synth.cpu_reference_config(nchunks=1, with_tables=False).binning)
    med, mad = eng.bootstrap_median(R)
    eng.close()
    omed = ob.median(R)
    assert np.array_equal(med, omed)
    X = R - omed
    for i in range(6):
        for j in range(i, 6):
            prod = X[:, i] * X[:, j]
            if np.isnan(prod).any():   # infinity times a zero deviation: no order, no median
                continue
            want = ob.median(prod[:, None])[0]
            assert mad[i, j] == want and mad[j, i] == want, (i, j)
