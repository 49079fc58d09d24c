"""The device spectrum at the edges of its passes: FFT lengths of one, two and three passes
(2^5 .. 2^9, 2^10 .. 2^18, 2^19 up), odd and even radices, odd and even lengths, no padding, against
the oracle's numpy FFT.

An FFT's amplitude is off by a few eps log2(L) times the largest amplitude (two transforms and the
chirps: under 10 eps log2(L)), the power by twice that: 20 * 2.2e-16 * 20 < 1e-13 at L = 2^20; the
test allows 4e-13 of the largest power."""
import numpy as np
import pytest

from ggbtddft_amd import spectrum as spec
from oracle import spectrum as OS

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,n_pad", [(16, 8), (17, 8), (33, 0), (256, 2), (257, 3), (513, 8), (2049, 1),
                                     (30840, 8), (131072, 1), (131073, 0), (300001, 1)])
def test_power_at_pass_edges(n, n_pad):
    print("case: spectrum passes n=%d n_pad=%d" % (n, n_pad), flush=True)
    rng = np.random.default_rng(n)
    x = rng.standard_normal(n)
    _, p_h = OS.acceleration_spectrum(x, 0.05, n_pad=n_pad)
    fits = spec.noalloc_fits(n, n_pad)
    _, p_d, _ = spec.device_spectrum(x, 0.05, n_pad=n_pad)
    assert p_d.shape == p_h.shape
    assert np.abs(p_d - p_h).max() <= 4e-13 * p_h.max()
    if fits:
        _, p_n, _ = spec.device_spectrum(x, 0.05, n_pad=n_pad, noalloc=True)
        assert np.array_equal(p_n, p_d)
