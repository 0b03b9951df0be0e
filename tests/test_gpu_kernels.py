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


def _wf(kind):
    from gwfast_amd.waveforms import IMRPhenomD, TaylorF2_RestrictedPN
    return {11: lambda: IMRPhenomD(), 12: lambda: TaylorF2_RestrictedPN(is_eccentric=True),
            13: lambda: TaylorF2_RestrictedPN(is_tidal=True),
            14: lambda: TaylorF2_RestrictedPN(is_tidal=True, is_eccentric=True)}[kind]()


def _events(P, n, seed):
    ev = (catalog.draw_bns if P in (13, 14) else catalog.draw_bbh)(n, seed=seed)
    if P in (12, 14):
        ev['ecc'] = np.random.default_rng(seed).uniform(0.01, 0.1, n)
    return ev


@pytest.mark.parametrize('P', [11, 12, 13, 14])
@pytest.mark.parametrize('res', [2, 64, 65, 200])
def test_block_products_against_single_arm_sums(P, res):
    """Per-arm matrices and the network sum (4 x 4 block products on the matrix
    cores) against the single-wave kernel's VALU sums, one launch per arm.  Both
    are FP64 sums of at most 200 points, so they differ by rounding: 1e-11 of
    sqrt(F_aa F_bb) is far above 200 ulp and far below any wrong element."""
    from tests._common import NET_C1, hip_net, norm_err
    from gwfast_amd import _engine as E, signal as S
    wf = _wf(P)
    rows = E.to_dev(E.param_rows(_events(P, 5, 3), P in (13, 14), P in (12, 14)))
    net = hip_net(wf, NET_C1, True)
    sigs = list(net.signals.values())
    one = np.stack([S.fisher_device(sigs, wf, rows, res, arm=a).cpu().numpy() for a in range(5)])
    arms = S.fisher_arms_device(sigs, wf, rows, res).cpu().numpy()
    total = net.fisher_device(rows, res).cpu().numpy()
    for a in range(5):
        assert norm_err(arms[a], one[a]) < 1e-11
    assert norm_err(total, one.sum(axis=0)) < 1e-11
