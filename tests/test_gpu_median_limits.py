"""The median bootstrap at the limits of its kernels (needs an MI355X): with
45 bands or more, 64 values are ranked as they are, up to 512, 2048 and 8192 are
counted in registers; fewer bands and longer columns take the radix select.  Bit for bit against a sort by
order-preserving keys: -0 before +0, NaN past the infinity of its sign."""
import numpy as np
import pytest

from lyspeq_amd import synth
from lyspeq_amd.qml import QMLEngine

pytestmark = pytest.mark.gpu


def _bits(x):
    return np.ascontiguousarray(x).view(np.int64)


def _median(x):
    """Of the values in key order: the middle one, or the half-sum of the two."""
    u = _bits(x)
    k = np.sort(np.where(u < 0, u ^ np.int64(2**63 - 1), u))
    v = np.where(k < 0, k ^ np.int64(2**63 - 1), k).view(np.float64)
    n = v.size
    return v[n // 2] if n % 2 else (v[n // 2 - 1] + v[n // 2]) / 2


def _run(R):
    eng = QMLEngine(synth.cpu_reference_config(nchunks=1, with_tables=False).binning)
    med, mad = eng.bootstrap_median(R)
    eng.close()
    return med, mad


def _widen(R, bands):
    """The columns again and again, times powers of two, up to so many."""
    n = R.shape[1]
    return np.concatenate([R * 2.0 ** k for k in range(max(1, -(-bands // n)))], axis=1)[:, :max(bands, n)]


def _check(R, bands=0, nan_products=False):
    """Every pair of R's columns; widened to more bands, some of the others too."""
    n, R = R.shape[1], _widen(R, bands)
    med, mad = _run(R)
    want = np.array([_median(r) for r in R.T])
    assert np.array_equal(_bits(med), _bits(want))
    X = np.ascontiguousarray(R.T) - want[:, None]
    T = len(X)
    pairs = [(i, j) for i in range(n) for j in range(i, n)]
    pairs += [tuple(sorted(p)) for p in np.random.default_rng(T).integers(0, T, (40 if T > n else 0, 2))]
    for i, j in pairs:
        p = X[i] * X[j]
        if nan_products and np.isnan(p).any():      # infinity times zero: the sign of that NaN is the machine's
            continue
        assert _bits(mad[i, j]) == _bits(_median(p)) == _bits(mad[j, i]), (i, j)


@pytest.mark.parametrize("bands", [0, 45])
@pytest.mark.parametrize("nboots", [63, 64, 65, 511, 512, 513, 2047, 2048, 2049, 8191, 8192, 8193, 20480, 20481])
def test_counts_of_realisations(nboots, bands):
    print(f"[case] median limits {nboots} {bands}", flush=True)
    rng = np.random.default_rng(nboots)
    R = rng.standard_normal((nboots, 6))
    R[:, 1] = np.exp(8 * R[:, 1])                              # many decades
    R[:, 2] = np.sort(R[:, 2])                                 # an order the sample follows
    R[:, 3] = np.where(R[:, 3] > 1.5, np.nan, R[:, 3])         # NaN past the rank
    R[:, 4] = np.where(np.arange(nboots) % 61 == 0, np.nan, R[:, 4] ** 3)
    R[:, 5] += 0.7 * R[:, 0]
    _check(R, bands)


@pytest.mark.parametrize("T", [1, 7, 8, 9, 15, 16, 17, 24, 25, 33, 44, 45, 56, 57])
def test_band_pairs(T):
    """Every pair of the folded triangle, at whole and partial eights of bands."""
    print(f"[case] median of {T} bands", flush=True)
    _check(np.random.default_rng(T).standard_normal((70, T)))


@pytest.mark.parametrize("bands", [0, 48])
@pytest.mark.parametrize("nboots", [66, 101, 512, 513, 2000, 2049, 8000, 8191, 8194])
def test_equal_values(nboots, bands):
    """Columns whose median has many copies: whole and tenth values, one value,
    zeros of both signs, two values that part the two ranks or nearly so, a value
    repeated at few places, infinities on both sides and on the median."""
    print(f"[case] median of equal values {nboots} {bands}", flush=True)
    rng = np.random.default_rng(nboots + 1)
    g = rng.standard_normal((nboots, 12))
    n = np.arange(nboots)
    R = g.copy()
    R[:, 0] = np.round(g[:, 0])
    R[:, 1] = np.round(g[:, 1], 1)
    R[:, 2] = 3.25
    R[:, 3] = np.copysign(0.0, g[:, 3])
    R[:, 4] = np.where(np.abs(g[:, 4]) < 0.5, np.copysign(0.0, g[:, 5]), g[:, 4])
    R[:, 5] = np.where(n < nboots // 2, -1.0, 2.0)             # one value for each rank where nboots is even
    R[:, 6] = np.where(n < nboots // 2 + 1, -1.0, 2.0)
    R[:, 7] = np.where(n % 50 == 3, np.median(g[:, 7]), g[:, 7])
    R[:, 8] = rng.poisson(1.0, nboots)
    R[:, 9] = np.where(np.abs(g[:, 9]) > 1.2, np.copysign(np.inf, g[:, 9]), np.abs(g[:, 9]) + 1.0)
    R[:, 10] = np.round(g[:, 10], 2)
    R[:, 11] = np.exp(6 * np.round(g[:, 11], 1))
    _check(R, bands, nan_products=True)


def test_infinite_medians():
    """A median among equal infinities, on its own."""
    print("[case] infinite medians", flush=True)
    for nboots in (100, 3000):
        n = np.arange(nboots)
        R = np.stack([np.where(n % 3 == 0, 1.0 + n, np.inf), np.where(n % 3 == 0, 1.0 + n, -np.inf)], axis=1)
        for bands in (2, 46):
            med, _ = _run(_widen(R, bands))
            assert np.array_equal(med, np.tile([np.inf, -np.inf], bands // 2))
