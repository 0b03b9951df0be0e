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


@pytest.mark.parametrize('B', [1, 15, 17, 300, 513, 4097])
def test_network_passes_against_their_building_blocks(B):
    """The fused training passes at the edges of their 16-row workgroups and
    512-row ranges: y, Z and H bit for bit those of gwf_gemm_bf16,
    gwf_bias_silu and gwf_head_forward (same products in the same order);
    gradients against 64-bit sums of the building blocks' bf16 dZ and H, within
    B roundings of 2^-24 of the sum of moduli."""
    import ctypes
    import torch
    from gwfast_amd import _engine as E, _native as N, screen
    sc = screen.SNRScreen(seed=2)
    rng = np.random.default_rng(B)
    theta = sc.params()
    theta[screen.OFFSETS['b1'][0]:] = rng.normal(0., 0.2, screen.N_PARAMS - screen.OFFSETS['b1'][0])
    sc.set_params(theta)
    x = rng.normal(0., 1., (B, screen.KFEAT))
    x[:, screen.NFEAT:] = 0.
    X = torch.as_tensor(x, dtype=torch.float32).to(torch.bfloat16).cuda()
    g = torch.as_tensor(rng.normal(0., 1., B), dtype=torch.float32).cuda()
    y, bt = sc.forward_train(X)
    sc.backward(X, bt, g)
    grad = sc.grad.cpu().numpy().astype(np.float64)
    sc.backward(X, bt, g)
    assert np.array_equal(grad, sc.grad.cpu().numpy())

    p = lambda t: ctypes.c_void_p(t.data_ptr())
    v = lambda flat, name: p(sc._view(flat, name))
    s, HID = N.stream_ptr(), screen.HID
    new = lambda *shape: torch.empty(shape, dtype=torch.float32, device='cuda')
    newb = lambda: torch.empty((B, HID), dtype=torch.bfloat16, device='cuda')
    Z, H, inp, k = [], [], X, screen.KFEAT
    for l in '123':
        C, z, h = new(B, HID), new(B, HID), newb()
        E.call('gwf_gemm_bf16', B, HID, k, 1.0, p(inp), k, 1, v(sc.theta_bf, 'W' + l), 1, k, 0.0, p(C), HID, 1, s)
        E.call('gwf_bias_silu', p(C), v(sc.theta, 'b' + l), B, HID, p(z), p(h), s)
        Z.append(z)
        H.append(h)
        inp, k = h, HID
    yr = new(B)
    E.call('gwf_head_forward', p(H[2]), v(sc.theta, 'w4'), v(sc.theta, 'b4'), B, p(yr), s)
    assert torch.equal(y, yr)
    for l in range(3):
        assert torch.equal(bt.Z[l], Z[l]) and torch.equal(bt.H[l].view(torch.int16), H[l].view(torch.int16))

    def check(name, ref, moduli):
        o, n, shape = screen.OFFSETS[name]
        d = np.abs(grad[o:o + n].reshape(shape) - ref)
        assert np.all(d <= B * 2. ** -24 * moduli + 1e-30), (name, float(np.max(d)))

    f64 = lambda t: t.to(torch.float64).cpu().numpy()
    g64, h3 = f64(g), f64(H[2])
    check('b4', g64.sum(), np.abs(g64).sum())
    check('w4', g64 @ h3, np.abs(g64) @ np.abs(h3))
    dH = g[:, None] * sc._view(sc.theta, 'w4')[None, :]
    for l in (2, 1, 0):
        dZ, dZb = new(B, HID), newb()
        E.call('gwf_silu_backward', p(dH), p(Z[l]), B * HID, p(dZ), p(dZb), s)
        dz, dzb, hp = f64(dZ), f64(dZb), f64(H[l - 1] if l else X)
        check('b%d' % (l + 1), dz.sum(0), np.abs(dz).sum(0))
        check('W%d' % (l + 1), dzb.T @ hp, np.abs(dzb).T @ np.abs(hp))
        if l:
            dH = new(B, HID)
            E.call('gwf_gemm_bf16', B, HID, HID, 1.0, p(dZb), HID, 1, v(sc.theta_bf, 'W%d' % (l + 1)), HID, 1, 0.0,
                   p(dH), HID, 1, s)


@pytest.mark.parametrize('n', [1, 127, 129, 300])
def test_screen_is_the_same_for_every_batch_and_keeps_nan(n):
    """An event's prediction does not depend on the batch it is in (the
    128-event blocks' edges), and an event without a finite feature predicts
    NaN and is recomputed (class 1)."""
    import torch
    from gwfast_amd import _engine as E, screen
    rows = E.to_dev(E.param_rows(catalog.draw_bbh(1000, seed=9), False))
    sc = screen.SNRScreen(seed=3)
    sc.fit_normalisation(rows, torch.zeros(1000, dtype=torch.float64))
    few = rows[:, :n].contiguous()
    assert torch.equal(sc.predict_log_snr(few), sc.predict_log_snr(rows)[:n])
    for value in (float('nan'), float('inf'), 0.):
        few[2, n - 1] = value
        ls = sc.predict_log_snr(few)
        assert bool(torch.isnan(ls[n - 1])) and bool(torch.isfinite(ls[:n - 1]).all())
        assert int(sc.classify(few)[n - 1]) == 1


@pytest.mark.parametrize('P', [11, 12, 13, 14])
@pytest.mark.parametrize('n,nf', [(1, 1), (5, 63), (3, 64), (9, 192), (17, 193), (8, 257), (66, 1000)])
def test_gram_over_an_events_waves(P, n, nf):
    """The plain Gram, one wave or four per event, against torch in FP64: sums
    of 2 nf products, so 4 nf 2^-52 of the sums of moduli."""
    import torch
    from gwfast_amd import _engine as E, signal as S
    rng = np.random.default_rng(nf)
    J, f = rng.standard_normal((P, n, nf, 2)), np.sort(rng.uniform(1., 9., (nf, n)), axis=0)
    psd = rng.uniform(0.5, 2., (nf, n))
    got = S.gram_device(E.to_dev(J), E.to_dev(f), E.to_dev(psd), P)
    twice = S.gram_device(E.to_dev(J), E.to_dev(f), E.to_dev(psd), P, out=got.clone(), accumulate=True)
    w = np.zeros_like(f)
    w[1:] += 0.5 * np.diff(f, axis=0)
    w[:-1] += 0.5 * np.diff(f, axis=0)
    x = J * np.sqrt(4. * w / psd).T[None, :, :, None]
    x = x.reshape(P, n, -1).transpose(1, 0, 2)
    ref, mod = x @ x.transpose(0, 2, 1), np.abs(x) @ np.abs(x).transpose(0, 2, 1)
    d = np.abs(got.cpu().numpy().transpose(2, 0, 1) - ref)
    assert np.all(d <= 4 * nf * 2. ** -52 * mod + 1e-300)
    assert torch.equal(twice, 2 * got)


@pytest.mark.parametrize('P', [1, 3, 4, 6, 11, 12, 13, 14, 16])
@pytest.mark.parametrize('n,nf', [(1, 1), (3, 255), (9, 256), (17, 700)])
def test_strain_vjp_at_any_parameter_count(P, n, nf):
    """g_p = sum_f Re(conj(gh) J_p) against numpy in FP64 (4 nf 2^-52 of the
    sum of moduli; the tcoal row scaled)."""
    import torch
    from gwfast_amd import _engine as E, _native as N
    rng = np.random.default_rng(nf)
    J, gh = rng.standard_normal((P, n, nf, 2)), rng.standard_normal((nf, n, 2))
    Jd, gd, g = E.to_dev(J), E.to_dev(gh), torch.empty((P, n), dtype=torch.float64, device='cuda')
    E.call('gwf_strain_vjp', N.ptr(Jd), N.ptr(gd), P, n, nf, 86400.0, N.ptr(g), N.stream_ptr())
    s = np.ones((P, 1))
    s[7:8] = 86400.
    prod = J * gh.transpose(1, 0, 2)[None]
    d = np.abs(g.cpu().numpy() - s * prod.sum(axis=(2, 3)))
    assert np.all(d <= 4 * nf * 2. ** -52 * s * np.abs(prod).sum(axis=(2, 3)))


@pytest.mark.parametrize('P', [11, 13])
@pytest.mark.parametrize('n,nf', [(1, 1), (1, 64), (3, 130), (3, 500)])
def test_strain_split_over_an_events_points(P, n, nf):
    """Few events, their points spread over many waves, against the same
    events among 9000 (one wave each): bit for bit."""
    from tests._common import NET_C0, hip_net
    from gwfast_amd import _engine as E, signal as S
    wf = _wf(P)
    rows = E.to_dev(E.param_rows(_events(P, n, 6), P == 13))
    f = E.to_dev(np.geomspace(np.full(n, 3.), np.full(n, 50.), nf))
    sig = list(hip_net(wf, NET_C0, True).signals.values())[0]
    k = 9000 // n
    h, J = S.strain_device(sig, rows, f, 0)
    hm, Jm = S.strain_device(sig, rows.repeat(1, k).contiguous(), f.repeat(1, k).contiguous(), 0)
    assert np.array_equal(h.cpu().numpy(), hm[:, :n].cpu().numpy())
    assert np.array_equal(J.cpu().numpy(), Jm[:, :n].cpu().numpy())


SITES_10_ARMS = ['ETS', 'ETMR', 'CE1Id', 'CE2NM', 'Virgo', 'KAGRA']


@pytest.mark.parametrize('P', [11, 12, 13, 'NRTidalv2'])
@pytest.mark.parametrize('arms', [5, 10])
@pytest.mark.parametrize('res', [2, 64, 65, 513, 1000])
def test_snr_of_few_and_many_events(P, arms, res):
    """Few events (a block of eight waves each, up to 8 arms) against the same
    events among 1000 (a wave each), and the SNR's own records against those a
    caller prepares for the Fisher kernels: the same terms in the same order up
    to the compiler's contractions, a few ulp of each, so 10^3 2^-52 relative."""
    import torch
    from tests._common import NET_C1, hip_net
    from gwfast_amd import _engine as E, _native as N, gwfastGlobals as glob, signal as S
    from gwfast_amd.waveforms import IMRPhenomD_NRTidalv2
    wf = IMRPhenomD_NRTidalv2() if P == 'NRTidalv2' else _wf(P)
    tidal = P in (13, 'NRTidalv2')
    n = 5
    rows = E.to_dev(E.param_rows(_events(13 if tidal else P, n, 8), tidal, P == 12))
    net = NET_C1 if arms == 5 else [(s, glob.PSD_ET if s[0] == 'E' else glob.PSD_CE) for s in SITES_10_ARMS]
    sigs = list(hip_net(wf, net, True).signals.values())
    few_len = np.array([res, 2, 64, max(2, res // 2), res], dtype=np.int32)

    def close(a, b):
        return bool(((a - b).abs() <= 1e3 * 2. ** -52 * b).all())

    for ln, tile in ((res, False), (few_len, True)):
        few = S.snr_sq_device(sigs, rows, ln)
        many = S.snr_sq_device(sigs, rows.repeat(1, 200).contiguous(), np.tile(ln, 200) if tile else ln)
        assert few.shape == (arms, n) and close(few, many[:, :n])
    ws, nb = E.workspace(n)
    dets = S._dets(sigs)
    E.call('gwf_prepare', wf.c_struct(), dets, len(sigs), N.ptr(rows), rows.stride(0), n, res, N.ptr(ws), nb,
           N.stream_ptr())
    out = torch.empty((arms, n), dtype=torch.float64, device='cuda')
    E.call('gwf_snr_prepared', wf.c_struct(), dets, len(sigs), n, res, N.ptr(out), N.ptr(ws), nb, N.stream_ptr())
    assert close(S.snr_sq_device(sigs, rows, res), out)


@pytest.mark.parametrize('n,longest', [(1025, 2), (1026, 64), (2600, 700), (3000, 65)])
def test_ragged_order_changes_no_result(n, longest):
    """A ragged batch taken longest first (a workspace with room for the order)
    and as it comes (one of the records and counters alone): bit for bit the
    same matrices, whatever the spread of the lengths."""
    import torch
    from tests._common import NET_C1, hip_net
    from gwfast_amd import _engine as E, _native as N, signal as S
    wf = _wf(11)
    rows = E.to_dev(E.param_rows(_events(11, n, 2), False))
    lengths = E.to_dev(np.random.default_rng(n).integers(2, longest + 1, n).astype(np.int32), torch.int32)
    sigs = list(hip_net(wf, NET_C1, True).signals.values())
    full = int(N.lib().gwf_workspace_bytes(n))
    ws = torch.empty(full, dtype=torch.uint8, device='cuda')
    out = []
    for size in (full, full - 4 * n):
        F = torch.full((11, 11, n), float('nan'), dtype=torch.float64, device='cuda')
        E.call('gwf_fisher_ragged', wf.c_struct(), S._dets(sigs), len(sigs), N.ptr(rows), rows.stride(0), n,
               N.ptr(lengths), -1, N.ptr(F), N.ptr(ws), size, N.stream_ptr())
        out.append(F.cpu().numpy())
    assert np.isfinite(out[0]).all() and np.array_equal(out[0], out[1])


@pytest.mark.parametrize('n', [1, 17, 300])
@pytest.mark.parametrize('nf', [1, 2, 12, 13, 24, 25, 80])
def test_grid_minimum_on_short_grids(n, nf):
    """The same on grids that the setup's lanes look through themselves and
    just longer ones: IMRPhenomD, NRTidalv2 and eccentric TaylorF2 bit for bit
    as with the reference frequency set to the minimum."""
    from gwfast_amd.waveforms import IMRPhenomD, IMRPhenomD_NRTidalv2, TaylorF2_RestrictedPN
    rng = np.random.default_rng(7)
    f = rng.uniform(5., 60., (nf, n))
    f[rng.integers(0, nf, n), np.arange(n)] = 4.5
    if nf > 1:
        f[(np.argmin(f, axis=0) + 1) % nf, np.arange(n)] = np.nan
    for make, key, P in ((IMRPhenomD, 'fRef', 11), (IMRPhenomD_NRTidalv2, 'fRef', 13),
                         (lambda **k: TaylorF2_RestrictedPN(is_eccentric=True, **k), 'fRef_ecc', 12)):
        ev = _events(P, n, 5)
        got, want = make().Phi(f, **ev), make(**{key: 4.5}).Phi(f, **ev)
        assert np.array_equal(got, want, equal_nan=True) and np.isfinite(got[np.isfinite(f)]).all()


# z and SiLU(z): past the exponential's overflow (-88.72) the quotient is -0, -inf / inf has no value
SILU_EXTREMES = [(-3.0e38, -0.), (-1e30, -0.), (-1e10, -0.), (-1000., -0.), (-100., -0.), (0., 0.), (-0., -0.),
                 (80., 80.), (1000., 1000.), (1e30, 1e30), (3.0e38, 3.0e38), (np.inf, np.inf), (-np.inf, np.nan),
                 (np.nan, np.nan)]


def test_silu_over_the_whole_range():
    """gwf_bias_silu against z / (1 + exp(-z)) in FP64.  The result is a bf16
    number (2^-8 of it covers its rounding and the FP32 exponential's error,
    below 2^-16 at |z| < 89); past the exponential's overflow the quotient is
    0, which is off by no more than 88.8 exp(-88.7) = 2.7e-37.  The extremes
    exactly."""
    import torch
    from gwfast_amd import _engine as E, _native as N
    z = np.concatenate([np.linspace(-95., 95., 4001), -np.geomspace(1e-6, 3e38, 1000), np.geomspace(1e-6, 3e38, 1000)])
    ext = np.array(SILU_EXTREMES, dtype=np.float32)
    zf = np.concatenate([z.astype(np.float32), ext[:, 0]])
    C = torch.as_tensor(zf, device='cuda').contiguous()
    zero = torch.zeros(1, dtype=torch.float32, device='cuda')
    H = torch.empty(zf.size, dtype=torch.bfloat16, device='cuda')
    E.call('gwf_bias_silu', N.ptr(C), N.ptr(zero), zf.size, 1, None, N.ptr(H), N.stream_ptr())
    h = H.to(torch.float64).cpu().numpy()
    z64 = zf[:z.size].astype(np.float64)
    with np.errstate(over='ignore'):
        ref = z64 / (1. + np.exp(-z64))
    assert np.all(np.abs(h[:z.size] - ref) <= 2. ** -8 * np.abs(ref) + 2.7e-37)
    want = torch.as_tensor(ext[:, 1]).to(torch.bfloat16).to(torch.float64).numpy()
    assert np.array_equal(h[z.size:], want, equal_nan=True)


@pytest.mark.parametrize('unit', [0, 63, 64, 255])
def test_a_saturated_unit_is_the_same_in_training_and_screen(unit):
    """One unit far below and far above the exponential's range in every
    layer, and one of infinite activation: the screen's prediction, the
    training forward's and, for the finite ones, 64-bit arithmetic on the same
    bf16 weights (the saturated unit's SiLU is -0, or the unit itself) agree."""
    import torch
    from gwfast_amd import _engine as E, screen
    n = 200
    rows = E.to_dev(E.param_rows(catalog.draw_bbh(n, seed=4), False))
    for bias, value in ((-1e30, 0.), (-3e38, 0.), (-90., 0.), (np.inf, np.inf)):
        sc = screen.SNRScreen(seed=1)
        sc.fit_normalisation(rows, torch.zeros(n, dtype=torch.float64))
        theta = sc.params()
        for b in ('b1', 'b2', 'b3'):
            theta[screen.OFFSETS[b][0] + unit] = bias
        if np.isinf(value):  # no products of the infinite unit but the output's
            for b in ('b1', 'b2'):
                theta[screen.OFFSETS[b][0] + unit] = 0.
            theta[screen.OFFSETS['w4'][0] + unit] = 1.
        sc.set_params(theta)
        y = sc.forward_train(sc.features(rows))[0].to(torch.float64).cpu().numpy()
        ls = sc.predict_log_snr(rows).to(torch.float64).cpu().numpy()
        if np.isinf(value):
            assert np.all(y == np.inf) and np.all(ls == np.inf) and int(sc.classify(rows).min()) == 2
            continue
        h = sc.features(rows).to(torch.float64).cpu().numpy()
        f64 = lambda flat, name: sc._view(flat, name).to(torch.float64).cpu().numpy()
        for l in '123':
            zl = h @ f64(sc.theta_bf, 'W' + l).T + f64(sc.theta, 'b' + l)
            with np.errstate(over='ignore'):
                hl = zl / (1. + np.exp(-zl))
            h = torch.as_tensor(hl).to(torch.bfloat16).to(torch.float64).numpy()
        ref = h @ f64(sc.theta, 'w4') + f64(sc.theta, 'b4')
        # activations differ by a bf16 rounding (2^-8) where FP32 and FP64 fall on two sides of a tie
        tol = 2. ** -8 * 3 * (np.abs(h) @ np.abs(f64(sc.theta, 'w4')) + np.abs(ref))
        assert np.all(np.abs(y - ref) <= tol) and np.all(np.abs(ls - y * sc.y_scale - sc.y_shift) <= tol)


def _models():
    from gwfast_amd.waveforms import IMRPhenomD_NRTidalv2
    return {11: lambda: _wf(11), 12: lambda: _wf(12), 13: lambda: _wf(13), 14: lambda: _wf(14),
            'NRTidalv2': lambda: IMRPhenomD_NRTidalv2()}


def _model_rows(P, n, seed):
    from gwfast_amd import _engine as E
    tidal = P in (13, 14, 'NRTidalv2')
    ev = _events(14 if P == 14 else (13 if tidal else P), n, seed)
    return E.to_dev(E.param_rows(ev, tidal, P in (12, 14)))


@pytest.mark.parametrize('P', [11, 12, 13, 14, 'NRTidalv2'])
@pytest.mark.parametrize('n', [1, 3, 300])
def test_snr_call_leaves_the_prepared_records(P, n):
    """gwf_snr and gwf_snr_ragged are gwf_prepare and the SNR of its records:
    the same SNR bit for bit, and a workspace (of NaN before) from which
    gwf_fisher_prepared gives gwf_fisher's matrices bit for bit."""
    import torch
    from tests._common import NET_C1, hip_net
    from gwfast_amd import _engine as E, _native as N, signal as S
    wf, rows, res = _models()[P](), _model_rows(P, n, 8), 130
    sigs = list(hip_net(wf, NET_C1, True).signals.values())
    dets, nd, s = S._dets(sigs), len(sigs), N.stream_ptr()
    nb = int(N.lib().gwf_workspace_bytes(n))
    lengths = torch.full((n,), res, dtype=torch.int32, device='cuda')
    F = S.fisher_device(sigs, wf, rows, res)

    def workspace():
        return torch.full((nb,), 0xff, dtype=torch.uint8, device='cuda')

    def prepared(ws, entry, extra=()):
        out = torch.empty(F.shape if entry == 'gwf_fisher_prepared' else (5, n), dtype=torch.float64, device='cuda')
        E.call(entry, wf.c_struct(), dets, nd, n, res, *extra, N.ptr(out), N.ptr(ws), nb, s)
        return out

    ws = workspace()
    E.call('gwf_prepare', wf.c_struct(), dets, nd, N.ptr(rows), rows.stride(0), n, res, N.ptr(ws), nb, s)
    snr = prepared(ws, 'gwf_snr_prepared')
    for entry, length in (('gwf_snr', res), ('gwf_snr_ragged', N.ptr(lengths))):
        ws, out = workspace(), torch.empty((5, n), dtype=torch.float64, device='cuda')
        E.call(entry, wf.c_struct(), dets, nd, N.ptr(rows), rows.stride(0), n, length, N.ptr(out), N.ptr(ws), nb, s)
        assert torch.equal(out, snr)
        assert torch.equal(prepared(ws, 'gwf_fisher_prepared', (-1,)), F)


@pytest.mark.parametrize('P', [11, 12, 13, 14, 'NRTidalv2'])
@pytest.mark.parametrize('motion', [True, False])
def test_records_of_the_snr_alone_give_no_fisher_matrix(P, motion):
    """gwf_snr_once's records: gwf_snr_prepared reads them like any, and the
    Fisher matrix of every event has NaN in it, whatever the records held
    before (those of gwf_prepare here), for network sums and single arms."""
    import torch
    from tests._common import NET_C1, hip_net
    from gwfast_amd import _engine as E, _native as N, signal as S
    wf, n, res = _models()[P](), 5, 130
    rows = _model_rows(P, n, 8)
    sigs = list(hip_net(wf, NET_C1, motion).signals.values())
    dets, nd, s = S._dets(sigs), len(sigs), N.stream_ptr()
    nb = int(N.lib().gwf_workspace_bytes(n))
    ws = torch.empty(nb, dtype=torch.uint8, device='cuda')
    for lengths in (None, torch.full((n,), res, dtype=torch.int32, device='cuda')):
        E.call('gwf_prepare', wf.c_struct(), dets, nd, N.ptr(rows), rows.stride(0), n, res, N.ptr(ws), nb, s)
        out, again = torch.empty((2, 5, n), dtype=torch.float64, device='cuda')
        E.call('gwf_snr_once', wf.c_struct(), dets, nd, N.ptr(rows), rows.stride(0), n, res, N.ptr(lengths),
               N.ptr(out), N.ptr(ws), nb, s)
        E.call('gwf_snr_prepared', wf.c_struct(), dets, nd, n, res, N.ptr(again), N.ptr(ws), nb, s)
        assert bool((out > 0).all()) and torch.equal(out, again)
        for arm in (-1, 0, 4):
            F = torch.empty((wf.nParams, wf.nParams, n), dtype=torch.float64, device='cuda')
            E.call('gwf_fisher_prepared', wf.c_struct(), dets, nd, n, res, arm, N.ptr(F), N.ptr(ws), nb, s)
            assert bool(torch.isnan(F[5]).all()) and bool(torch.isnan(F[:, 5]).all())
    assert S.snr_sq_device(sigs, rows[:, :0].contiguous(), np.zeros(0, dtype=np.int32)).shape == (5, 0)


@pytest.mark.parametrize('P', [11, 12, 13, 14, 'NRTidalv2'])
@pytest.mark.parametrize('sites', [1, 2, 3, 4, 6])
@pytest.mark.parametrize('res', [2, 63, 65, 513, 1000])
def test_snr_does_not_depend_on_the_batch(P, sites, res):
    """An event's SNR alone, among a few and among many (uniform and ragged
    grids): bit for bit, so that a catalogue in chunks of any size, or resumed
    in others, holds the same SNRs."""
    import torch
    from tests._common import hip_net
    from gwfast_amd import gwfastGlobals as glob, signal as S
    wf, n = _models()[P](), 7
    rows = _model_rows(P, n, 8)
    net = [(s, glob.PSD_ET if s[0] == 'E' else glob.PSD_CE) for s in ['CE1Id', 'ETS', 'CE2NM', 'Virgo', 'KAGRA', 'ETMR'][:sites]]
    sigs = list(hip_net(wf, net, True).signals.values())
    lengths = np.array([res, 2, 64, max(2, res // 2), res, 700, 129], dtype=np.int32)
    for ln in (res, lengths):
        pick = lambda i: ln if np.isscalar(ln) else ln[i:i + 1]
        many = S.snr_sq_device(sigs, rows.repeat(1, 200).contiguous(), ln if np.isscalar(ln) else np.tile(ln, 200))
        assert torch.equal(many, many[:, :n].repeat(1, 200))
        assert torch.equal(S.snr_sq_device(sigs, rows, ln), many[:, :n])
        for i in range(2):
            assert torch.equal(S.snr_sq_device(sigs, rows[:, i:i + 1].contiguous(), pick(i)), many[:, i:i + 1])


@pytest.mark.parametrize('n', [1025, 1500, 4096, 9001, 20011])
@pytest.mark.parametrize('kind', ['equal', 'narrow', 'wide', 'few long', 'longest unseen', 'out of range'])
def test_ragged_order_where_it_pays_and_where_not(n, kind):
    """The order is made by the spread of a sample of the lengths (every
    n // 4096-th group of 64): with it, without (a workspace of the records and
    counters alone) and for events by themselves the same matrices bit for bit,
    with the longest events in the sample or not and lengths below 2 (taken as
    2)."""
    import torch
    from tests._common import NET_C1, hip_net
    from gwfast_amd import _engine as E, _native as N, signal as S
    wf = _wf(11)
    rows = E.to_dev(E.param_rows(_events(11, 500, 2), False)).repeat(1, n // 500 + 1)[:, :n].contiguous()
    rng = np.random.default_rng(n)
    lengths = rng.integers(2, 130, n)
    if kind == 'equal':
        lengths[:] = 64
    elif kind == 'wide':
        lengths = rng.integers(2, 1500, n)
    elif kind == 'few long':
        lengths[rng.random(n) < 0.01] = 2000
    elif kind == 'longest unseen':
        lengths[::64] = 1500
        lengths[65:128] = 4000
    elif kind == 'out of range':
        lengths[::7], lengths[1::7], lengths[-1] = -5, 0, 1400
    sigs = list(hip_net(wf, NET_C1, True).signals.values())
    full = int(N.lib().gwf_workspace_bytes(n))
    ws = torch.full((full,), 0xff, dtype=torch.uint8, device='cuda')
    L = E.to_dev(lengths.astype(np.int32), torch.int32)
    out = []
    for size in (full, full - 4 * n):
        F = torch.full((11, 11, n), float('nan'), dtype=torch.float64, device='cuda')
        E.call('gwf_fisher_ragged', wf.c_struct(), S._dets(sigs), len(sigs), N.ptr(rows), rows.stride(0), n,
               N.ptr(L), -1, N.ptr(F), N.ptr(ws), size, N.stream_ptr())
        out.append(F)
    assert bool(torch.isfinite(out[0]).all()) and torch.equal(out[0], out[1])
    for e in (0, 1, 66, n - 1):
        one = S.fisher_device(sigs, wf, rows[:, e:e + 1].contiguous(), np.array([max(2, lengths[e])]))
        assert torch.equal(out[0][:, :, e], one[:, :, 0])


@pytest.mark.parametrize('P,line', [(11, 32768 // 4), ('NRTidalv2', 32768 // 6)])
def test_records_do_not_depend_on_the_batch(P, line):
    """The setup's constants take one of an event's lanes or one lane per event
    by the size of the batch: the same Fisher matrices bit for bit on both sides
    of the line."""
    import torch
    from tests._common import NET_C1, hip_net
    from gwfast_amd import signal as S
    wf, n = _models()[P](), 5
    rows = _model_rows(P, n, 8)
    sigs = list(hip_net(wf, NET_C1, True).signals.values())
    few = S.fisher_device(sigs, wf, rows, 70)
    for m in (line - 1, line, line + 1, 2 * line):
        many = S.fisher_device(sigs, wf, rows.repeat(1, m // n + 1)[:, :m].contiguous(), 70)
        assert torch.equal(many, few.repeat(1, 1, m // n + 1)[:, :, :m])


def test_captured_calls_follow_their_inputs():
    """The SNR alone, a ragged batch (once with an order and once without, by
    its lengths), strain rows with the grid's minimum and their VJP, recorded
    into one HIP graph: every replay on new inputs in the same buffers, with
    eager work between, gives the eager results bit for bit."""
    import torch
    from tests._common import NET_C1, hip_net
    from gwfast_amd import _engine as E, _native as N, signal as S
    wf, n, nf, res = _wf(11), 1200, 70, 130
    sigs = list(hip_net(wf, NET_C1, True).signals.values())
    dets, nd = S._dets(sigs), len(sigs)
    det = sigs[1].c_struct()
    nb = int(N.lib().gwf_workspace_bytes(n))
    new = lambda *shape: torch.empty(shape, dtype=torch.float64, device='cuda')
    wss = [torch.empty(nb, dtype=torch.uint8, device='cuda') for _ in range(3)]
    rows, f, gh = new(11, n), new(nf, n), new(nf, n, 2)
    lengths = torch.empty(n, dtype=torch.int32, device='cuda')
    out = {'snr': new(5, n), 'F': new(11, 11, n), 'h': new(nf, n, 2), 'J': new(11, n, nf, 2), 'g': new(11, n)}

    def calls():
        s = N.stream_ptr()
        E.call('gwf_snr_once', wf.c_struct(), dets, nd, N.ptr(rows), n, n, res, None, N.ptr(out['snr']), N.ptr(wss[0]), nb, s)
        E.call('gwf_fisher_ragged', wf.c_struct(), dets, nd, N.ptr(rows), n, n, N.ptr(lengths), -1, N.ptr(out['F']),
               N.ptr(wss[1]), nb, s)
        E.call('gwf_strain', wf.c_struct(), S.ctypes_byref(det), 0, N.ptr(rows), n, n, N.ptr(f), nf, N.ptr(out['h']),
               N.ptr(out['J']), N.ptr(wss[2]), nb, s)
        E.call('gwf_strain_vjp', N.ptr(out['J']), N.ptr(gh), 11, n, nf, 86400.0, N.ptr(out['g']), s)

    def fill(seed):
        rng = np.random.default_rng(seed)
        rows.copy_(E.to_dev(E.param_rows(_events(11, n, seed), False)))
        f.copy_(E.to_dev(np.sort(rng.uniform(4., 40., (nf, n)), axis=0)))
        gh.copy_(E.to_dev(rng.standard_normal((nf, n, 2))))
        lengths.copy_(E.to_dev(rng.integers(2, 1500 if seed % 2 else 100, n).astype(np.int32), torch.int32))

    fill(1)
    calls()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        calls()
    for seed in (2, 3, 4, 5):
        fill(seed)
        for o in out.values():
            o.fill_(float('nan'))
        graph.replay()
        got = {k: o.clone() for k, o in out.items()}
        calls()
        torch.cuda.synchronize()
        for k, o in out.items():
            assert bool(torch.isfinite(o).all()) and torch.equal(got[k], o), (k, seed)


@pytest.mark.parametrize('B', [300])
def test_captured_training_step_follows_its_inputs(B):
    """The training passes recorded into a HIP graph: every replay on new rows
    gives the eager predictions and gradients bit for bit."""
    import torch
    from gwfast_amd import screen
    sc = screen.SNRScreen(seed=4)
    gen = torch.Generator(device='cuda').manual_seed(1)
    X = torch.zeros((B, screen.KFEAT), dtype=torch.bfloat16, device='cuda')
    g = torch.empty(B, dtype=torch.float32, device='cuda')
    y, bt = sc.forward_train(X)

    def calls():
        sc.forward_train(X, bt)
        sc.backward(X, bt, g)

    def fill():
        X[:, :screen.NFEAT].copy_(torch.randn((B, screen.NFEAT), device='cuda', generator=gen))
        g.copy_(torch.randn(B, device='cuda', generator=gen))

    fill()
    calls()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        calls()
    for _ in range(3):
        fill()
        y.fill_(float('nan'))
        sc.grad.fill_(float('nan'))
        graph.replay()
        got = y.clone(), sc.grad.clone()
        calls()
        torch.cuda.synchronize()
        assert bool(torch.isfinite(y).all()) and torch.equal(got[0], y) and torch.equal(got[1], sc.grad)
