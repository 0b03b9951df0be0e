"""Kernels at the edges of their tiles, splits and ranges."""
import numpy as np
import pytest

from gwfast_amd import catalog

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('n,nf', [(1, 1), (1, 1023), (1, 5000), (3, 64), (4, 257), (15, 256), (16, 63), (33, 259)])
def test_grid_minimum_is_the_reference_frequency(n, nf):
    """IMRPhenomD without fRef takes each event's grid minimum, wherever it
    lies in the column: bit for bit the phase with fRef set to that value."""
    from gwfast_amd.waveforms import IMRPhenomD
    ev = catalog.draw_bbh(n, seed=5)
    rng = np.random.default_rng(6)
    f = rng.uniform(5., 60., (nf, n))
    f[rng.integers(0, nf, n), np.arange(n)] = 4.5
    if nf > 2:
        f[(np.argmin(f, axis=0) + 1) % nf, np.arange(n)] = np.nan  # a NaN is never the minimum
    got = IMRPhenomD().Phi(f, **ev)
    want = IMRPhenomD(fRef=4.5).Phi(f, **ev)
    assert np.array_equal(got, want, equal_nan=True)
    assert np.isfinite(got[np.isfinite(f)]).all()
