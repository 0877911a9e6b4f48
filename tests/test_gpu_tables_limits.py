"""The device signal tables at the limits of their grids (needs an MI355X)."""
import math

import numpy as np
import pytest
import torch

from lyspeq_amd import synth
from lyspeq_amd.qml import Binning, QMLEngine

pytestmark = pytest.mark.gpu

BINS = Binning(k0=0.0, nklin=10, dklin=0.002, nklog=0, dklog=0.1, z0=2.4, z_bin_width=0.2, nz=1, method=1,
               cont_logl_order=1, cont_lam_order=-1, max_forest_length_v=2.0e3)


def _columns(pair, nv, v_length, nz, cols, pd13):
    """Columns of the signal table by the inverse real FFT, modes with
    W^2 < 1e-40 left out."""
    n = 1 << (math.ceil(math.log2(4 * nv)) + 1)
    length = v_length / (nv - 1.0) / 2 * n
    k = np.arange(n // 2 + 1) * (2 * math.pi / length)
    R = synth.SPEED_OF_LIGHT / pair[0] / synth.ONE_SIGMA_2_FWHM
    w2 = synth.window_sq(k, pair[1], R)
    keep = np.arange(k.size) <= math.ceil(9.6 / (R * k[1]))
    zc, width = BINS.zbin_centers()[0], BINS.z_bin_width
    out = []
    for iz in cols:
        z = zc - width + width * (BINS.nz + 1) / (nz - 1.0) * iz
        f = np.zeros(k.size)
        f[keep] = w2[keep] * synth.pd13_power(k[keep], z, *pd13)
        out.append(np.fft.irfft(f, n)[:2 * nv:2] * n / length)
    return np.array(out).T


def test_more_than_2_31_modes_times_redshifts():
    """4097 velocities and 65535 redshifts: 32800 x 65536 elements of P_fid."""
    print("[case] 4097 x 65535 signal table", flush=True)
    pair, nv, v_length, nz = (2000, 50.0), 4097, 40960.0, 65535
    eng = QMLEngine(BINS)
    _, s = eng.make_tables([pair], nv, v_length, nz, synth.PD13_DEFAULT, deriv=False)
    eng.close()
    cols = [0, 1, 31, 32, 32767, 32768, 65533, 65534]
    want = _columns(pair, nv, v_length, nz, cols, synth.PD13_DEFAULT)
    assert np.max(np.abs(s[0][:, cols] - want)) < 1e-11 * np.max(np.abs(want))


def test_infinite_power_past_the_kept_modes():
    """1 + lambda k^2 is zero at k = 1/8, nine modes past the last kept one: a
    mode that is left out adds nothing, infinite or not."""
    print("[case] infinite power past the kept modes", flush=True)
    R_fwhm, nv, nz, mode = 1650, 1601, 3, 1975
    R = synth.SPEED_OF_LIGHT / R_fwhm / synth.ONE_SIGMA_2_FWHM
    n = 1 << (math.ceil(math.log2(4 * nv)) + 1)

    def step(v_length):
        return 2 * math.pi / (v_length / (nv - 1.0) / 2.0 * n)

    v_length = 2 * math.pi / (0.125 / mode) / n * 2 * (nv - 1)
    v_length = next(v for v in v_length + np.arange(-200, 200) * np.spacing(v_length) if mode * step(v) == 0.125)
    last = math.ceil(9.6 / (R * step(v_length)))
    assert last < mode < (last + 32) // 32 * 32     # in the last block of 32 modes
    pd13 = (0.066, -2.7, -0.1, 3.6, 0.0, -64.0)
    eng = QMLEngine(BINS)
    _, s = eng.make_tables([(R_fwhm, 50.0)], nv, v_length, nz, pd13, deriv=False)
    eng.close()
    want = _columns((R_fwhm, 50.0), nv, v_length, nz, range(nz), pd13)
    assert np.max(np.abs(s[0] - want)) < 1e-11 * np.max(np.abs(want))


@pytest.mark.parametrize("nv,nz", [(2, 2), (31, 15), (32, 16), (33, 17), (65, 31), (64, 32), (97, 33), (1601, 48),
                                   (1600, 49)])
def test_signal_blocks(nv, nz):
    """Velocities around the blocks of 32 and redshifts around those of 16 and
    32; a pair's table does not depend on the others of the call."""
    print(f"[case] signal blocks {nv} x {nz}", flush=True)
    pairs, v_length = [(2000, 50.0), (3100, 36.5), (4900, 65.9)], 10.0 * (nv - 1)
    eng = QMLEngine(BINS)
    _, s = eng.make_tables(pairs, nv, v_length, nz, synth.PD13_DEFAULT, deriv=False)
    _, one = eng.make_tables(pairs[1:2], nv, v_length, nz, synth.PD13_DEFAULT, deriv=False)
    eng.close()
    assert np.array_equal(s[1], one[0])
    for p, t in zip(pairs, s):
        want = _columns(p, nv, v_length, nz, range(nz), synth.PD13_DEFAULT)
        assert np.max(np.abs(t - want)) < 1e-11 * np.max(np.abs(want))


def test_scratch_of_a_large_table():
    """A signal table of 1.07 GB, whose P_fid grid takes 8.6 GB, is made with 14
    GB of device memory left: the sums need no further copies of the table."""
    print("[case] scratch of a large table", flush=True)
    pair, nv, v_length, nz = (2000, 50.0), 4097, 40960.0, 32767
    eng = QMLEngine(BINS)
    eng.make_tables([pair], 65, 640.0, 9, synth.PD13_DEFAULT)      # the kernels are loaded
    free = torch.cuda.mem_get_info()[0]
    held = torch.empty(free - (14 << 30), dtype=torch.uint8, device="cuda")
    try:
        _, s = eng.make_tables([pair], nv, v_length, nz, synth.PD13_DEFAULT, deriv=False)
    finally:
        del held
        torch.cuda.empty_cache()
        eng.close()
    want = _columns(pair, nv, v_length, nz, [0, nz - 1], synth.PD13_DEFAULT)
    assert np.max(np.abs(s[0][:, [0, nz - 1]] - want)) < 1e-11 * np.max(np.abs(want))
