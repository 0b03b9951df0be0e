"""The work a user of gwfast_amd has it do, as measurable cases.

Every case goes through the package's public entry points, with the event
populations of gwfast_amd.catalog, the detector sites and noise curves the
package ships, and sizes taken from bench.py, the tests and the tutorial the
package follows (100 events on 1000-point grids; catalogues of 10^4 to 10^6
events on 1000- to 2000-point grids).  A case's "kind" names the call:

  fisher_call   DetNet.FisherMatr on a dictionary of host arrays
  snr_call      DetNet.SNR on a dictionary of host arrays
  fisher        DetNet.fisher_device on rows that stay on the GPU, one grid
                length or (ragged) one per event
  fisher_arms   signal.fisher_arms_device: every arm's matrix, what
                FisherMatr(return_all=True) and the catalogue driver ask for
  fisher_duty   signal.fisher_masked_device: the duty-cycled network sum
  snr           DetNet.snr_device
  strain_grad   autodiff.strain, forward and backward of a data misfit
  derivatives   signal.strain_device + signal.gram_device: strain, derivative
                rows and their Fisher integral, what
                FisherMatr(return_derivatives=True) runs
  covariance    fisherTools.cov_device on a batch of Fisher matrices
  screen        SNRScreen.predict_log_snr
  screen_step   SNRScreen.forward_train + backward: one training step's
                prediction and gradients
"""
import math

import numpy as np
import torch

from gwfast_amd import _engine as E
from gwfast_amd import autodiff, catalog, fisherTools, gwfastGlobals as glob, screen, signal
from gwfast_amd.network import DetNet
from gwfast_amd.signal import GWSignal
from gwfast_amd.waveforms import IMRPhenomD, IMRPhenomD_NRTidalv2, TaylorF2_RestrictedPN

NETS = {
    'CE1Id': [('CE1Id', 'CE')],
    'ETS': [('ETS', 'ET')],
    '2CE': [('CE1Id', 'CE'), ('CE2NM', 'CE')],
    'ETS+2CE': [('ETS', 'ET'), ('CE1Id', 'CE'), ('CE2NM', 'CE')],
    'ETS+ETMRL+CE1Id': [('ETS', 'ET'), ('ETMRL45d', 'ET'), ('CE1Id', 'CE')],
}
PSD = {'ET': glob.PSD_ET, 'CE': glob.PSD_CE}
MODELS = {
    'IMRPhenomD': IMRPhenomD,
    'IMRPhenomD_NRTidalv2': IMRPhenomD_NRTidalv2,
    'TaylorF2': TaylorF2_RestrictedPN,
    'TaylorF2_tidal': lambda: TaylorF2_RestrictedPN(is_tidal=True),
    'TaylorF2_tidal_Kerr': lambda: TaylorF2_RestrictedPN(is_tidal=True, which_ISCO='Kerr'),
}
N_PAR = {'IMRPhenomD': 11, 'TaylorF2': 11, 'IMRPhenomD_NRTidalv2': 13, 'TaylorF2_tidal': 13,
         'TaylorF2_tidal_Kerr': 13}
ROW_NAMES = ('Mc', 'eta', 'dL', 'theta', 'phi', 'iota', 'psi', 'tcoal', 'Phicoal', 'chi1z', 'chi2z')
WAVE_KINDS = ('fisher_call', 'snr_call', 'fisher', 'fisher_arms', 'fisher_duty', 'snr', 'strain_grad', 'derivatives')


def _case(kind, name=None, **kw):
    c = {'kind': kind, **kw}
    if name is not None:
        c['name'] = name
    return c


def _wave(kind, model, net, n, res, name=None, motion=True, **kw):
    return _case(kind, name=name, model=model, net=net, n=n, res=res, motion=motion, **kw)


def listed():
    return [
        # one black-hole binary looked at by itself: the interactive call, all latency
        _wave('fisher_call', 'IMRPhenomD', 'ETS+2CE', 1, 1000, name='fisher_call_one_bbh'),
        # the tutorial's two calls: SNR and Fisher of 100 tidal binaries in the triangle
        _wave('snr_call', 'TaylorF2_tidal', 'ETS', 100, 1000, name='snr_call_tutorial_100'),
        _wave('fisher_call', 'TaylorF2_tidal', 'ETS', 100, 1000, name='fisher_call_tutorial_100'),
        # the benchmark's step: 10^4 black-hole binaries, parameters resident on the GPU
        _wave('fisher', 'IMRPhenomD', 'ETS+2CE', 10000, 2000, name='fisher_bbh_1e4', ragged=False),
        # neutron-star binaries whose grids follow their length in band
        _wave('fisher', 'TaylorF2_tidal_Kerr', 'ETS+2CE', 20000, 10000, name='fisher_ragged_bns_2e4', ragged=True),
        # one chunk of the catalogue driver, which keeps every arm's matrix (odd size: what passed the threshold)
        _wave('fisher_arms', 'IMRPhenomD_NRTidalv2', 'ETS+2CE', 3001, 1000, name='fisher_arms_bns_3001'),
        # the SNR pass over a catalogue before its threshold
        _wave('snr', 'IMRPhenomD', 'ETS+2CE', 100000, 1000, name='snr_bbh_1e5'),
        # gradients of a misfit through the strain, as an optimiser or sampler takes them
        _wave('strain_grad', 'IMRPhenomD', 'CE1Id', 500, 2000, name='strain_grad_500'),
        # derivative rows kept, and the Fisher integral over them
        _wave('derivatives', 'TaylorF2', 'CE1Id', 2000, 1000, name='derivatives_2000'),
        # covariances of a detected catalogue
        _case('covariance', name='covariance_2e4', n_par=11, n=20000),
        # the learned screen over a large catalogue, and one step of its training
        _case('screen', name='screen_1e6', n=1000000),
        _case('screen_step', name='screen_step_4096', n=4096),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the same calls: sizes over the whole range (over its
    logarithm), never dearer than the largest listed case."""
    kind = rng.choice(('fisher_call', 'snr_call', 'fisher', 'fisher', 'fisher_arms', 'fisher_duty', 'snr',
                       'strain_grad', 'derivatives', 'covariance', 'screen', 'screen_step'))
    if kind == 'covariance':
        return _case(kind, n_par=rng.choice((11, 11, 13)), n=_log_int(rng, 10, 50000))
    if kind == 'screen':
        return _case(kind, n=_log_int(rng, 1000, 1000000))
    if kind == 'screen_step':
        return _case(kind, n=_log_int(rng, 256, 8192))
    model = rng.choice(('IMRPhenomD', 'IMRPhenomD', 'IMRPhenomD_NRTidalv2', 'TaylorF2', 'TaylorF2_tidal'))
    net = rng.choice(tuple(NETS))
    motion = rng.random() < 0.8
    res = _log_int(rng, 200, 4000)
    if kind in ('fisher_call', 'snr_call'):
        return _wave(kind, model, net, _log_int(rng, 1, 1000), res, motion=motion)
    if kind == 'strain_grad':
        return _wave(kind, model, rng.choice(('CE1Id', 'ETS')), _log_int(rng, 1, 1000), min(res, 2000), motion=motion)
    if kind == 'derivatives':
        return _wave(kind, model, rng.choice(('CE1Id', 'ETS')), _log_int(rng, 10, 2000), min(res, 1500), motion=motion)
    if kind == 'snr':
        return _wave(kind, model, net, min(_log_int(rng, 10, 100000), int(1e8 / res)), res, motion=motion)
    if kind == 'fisher':
        ragged = rng.random() < 0.4
        return _wave(kind, model, net, min(_log_int(rng, 10, 30000), int(2e7 / res)), res, motion=motion, ragged=ragged)
    return _wave(kind, model, net, min(_log_int(rng, 10, 10000), int(1e7 / res)), res, motion=motion)


# ------------------------------------------------------------------ inputs
def _events(case, seed):
    bns = case['model'] in ('TaylorF2_tidal', 'TaylorF2_tidal_Kerr', 'IMRPhenomD_NRTidalv2')
    ev = (catalog.draw_bns if bns else catalog.draw_bbh)(case['n'], seed=seed)
    return ev, bns


def _network(case):
    wf = MODELS[case['model']]()
    sigs = {}
    for name, psd in NETS[case['net']]:
        d = glob.detectors[name]
        sigs[name] = GWSignal(wf, psd_path=PSD[psd], detector_shape=d['shape'], det_lat=d['lat'], det_long=d['long'],
                              det_xax=d['xax'], useEarthMotion=case['motion'], fmin=2., verbose=False)
    return wf, DetNet(sigs, verbose=False)


def _grid_lengths(case, seed):
    """Grid lengths of a ragged batch, uniform in [res / 20, res]."""
    return np.random.default_rng(seed + 1).integers(max(2, case['res'] // 20), case['res'] + 1, case['n']).astype(np.int32)


def _misfit_inputs(case, seed):
    """A fixed frequency grid below every event's cut and the weights of the
    misfit's gradient, (N_f, N_ev, 2)."""
    rng = np.random.default_rng(seed + 2)
    hi = rng.uniform(40., 60., case['n'])
    f = np.geomspace(np.full(case['n'], 2.), hi, case['res'])
    return f, rng.standard_normal((case['res'], case['n'], 2))


def _duty_masks(case, seed):
    n_arms = [3 if glob.detectors[name]['shape'] == 'T' else 1 for name, _ in NETS[case['net']]]
    rng = np.random.default_rng(seed + 3)
    return [(rng.random((k, case['n'])) < 0.85).astype(np.int64) for k in n_arms]


def _fisher_batch(case, seed):
    """Positive-definite matrices with the scales and the correlations that
    Fisher matrices of compact binaries have: condition numbers of the scaled
    matrix from 10^2 to 10^8, diagonals over many decades."""
    P, n = case['n_par'], case['n']
    rng = np.random.default_rng(seed)
    q, _ = np.linalg.qr(rng.standard_normal((n, P, P)))
    lam = 10. ** (-rng.uniform(2., 8., (n, 1)) * np.linspace(0., 1., P))
    A = np.einsum('nij,nj,nkj->nik', q, lam, q)
    s = 10. ** rng.uniform(-2., 5., (n, P))
    A = A * s[:, :, None] * s[:, None, :]
    A = 0.5 * (A + A.transpose(0, 2, 1))
    return np.ascontiguousarray(A.transpose(1, 2, 0))


def _screen_inputs(case, seed):
    ev = catalog.draw_bbh(case['n'], seed=seed)
    rng = np.random.default_rng(seed + 4)
    proxy = 5. - np.log(ev['dL']) + 0.2 * rng.standard_normal(case['n'])   # a log-SNR-like target
    return ev, proxy


def _screen_state(case, seed):
    ev, proxy = _screen_inputs(case, seed)
    rows = E.to_dev(E.param_rows(ev, False))
    sc = screen.SNRScreen(seed=seed)
    sc.fit_normalisation(rows, torch.from_numpy(proxy))
    return rows, sc, proxy


def prepare(case, seed):
    kind = case['kind']
    if kind == 'covariance':
        return {'kind': kind, 'F': E.to_dev(_fisher_batch(case, seed))}
    if kind == 'screen':
        rows, sc, _ = _screen_state(case, seed)
        return {'kind': kind, 'rows': rows, 'screen': sc}
    if kind == 'screen_step':
        rows, sc, proxy = _screen_state(case, seed)
        target = E.to_dev(((proxy - sc.y_shift) / sc.y_scale).astype(np.float32), torch.float32)
        return {'kind': kind, 'screen': sc, 'X': sc.features(rows), 'target': target}
    wf, net = _network(case)
    ev, bns = _events(case, seed)
    state = {'kind': kind, 'wf': wf, 'net': net, 'sigs': list(net.signals.values()), 'res': case['res'], 'ev': ev}
    if kind in ('fisher_call', 'snr_call'):
        return state
    state['rows'] = E.to_dev(E.param_rows(ev, bns))
    if kind == 'fisher' and case['ragged']:
        state['res'] = _grid_lengths(case, seed)
    if kind == 'fisher_duty':
        state['words'] = signal.mask_words(_duty_masks(case, seed))
    if kind == 'strain_grad':
        f, w = _misfit_inputs(case, seed)
        state['rows'].requires_grad_(True)
        state['f'], state['weights'] = E.to_dev(f), E.to_dev(w)
    if kind == 'derivatives':
        state['f'], state['S'] = signal.grid_device(state['sigs'][0], state['rows'], case['res'])
    return state


# -------------------------------------------------------------------- runs
def run(state):
    kind = state['kind']
    if kind == 'fisher_call':
        return state['net'].FisherMatr(dict(state['ev']), res=state['res'])
    if kind == 'snr_call':
        return state['net'].SNR(dict(state['ev']), res=state['res'])
    if kind == 'fisher':
        return state['net'].fisher_device(state['rows'], state['res'])
    if kind == 'fisher_arms':
        return signal.fisher_arms_device(state['sigs'], state['wf'], state['rows'], state['res'])
    if kind == 'fisher_duty':
        return signal.fisher_masked_device(state['sigs'], state['wf'], state['rows'], state['res'], state['words'])
    if kind == 'snr':
        return state['net'].snr_device(state['rows'], state['res'])
    if kind == 'strain_grad':
        rows = state['rows']
        h = autodiff.strain(state['sigs'][0], rows, state['f'], 0)
        (g,) = torch.autograd.grad(h, rows, grad_outputs=state['weights'])
        return h.detach(), g
    if kind == 'derivatives':
        h, J = signal.strain_device(state['sigs'][0], state['rows'], state['f'], 0)
        return h, J, signal.gram_device(J, state['f'], state['S'], state['wf'].nParams)
    if kind == 'covariance':
        C, _, cond, method = fisherTools.cov_device(state['F'])
        return C, cond, method
    if kind == 'screen':
        return state['screen'].predict_log_snr(state['rows'])
    sc = state['screen']
    y, bt = sc.forward_train(state['X'])
    sc.backward(state['X'], bt, (y - state['target']) * (2.0 / y.shape[0]))
    return y, sc.grad


# -------------------------------------------------------------------- work
def _n_arms(case):
    return sum(3 if glob.detectors[name]['shape'] == 'T' else 1 for name, _ in NETS[case['net']])


def work(case):
    """Inputs read once, outputs written once, and the arithmetic of the
    contraction each call ends in (a Fisher matrix: the upper triangle of
    P x P complex products per frequency and arm; an SNR: one squared
    modulus per frequency and arm); waveforms and projections come on top."""
    kind, n = case['kind'], case['n']
    if kind == 'covariance':
        P = case['n_par']
        return {'bytes': 8. * n * (2 * P * P + 1.5), 'flops': n * 2. * P ** 3}
    if kind in ('screen', 'screen_step'):
        fl = float(screen.FLOP_PER_INFERENCE) * n
        if kind == 'screen':
            return {'bytes': n * (11 * 8. + 4.) + 2. * screen.N_PARAMS, 'flops': fl}
        return {'bytes': n * (16 * 2. + 8.) + 6. * screen.N_PARAMS, 'flops': 3. * fl}
    P = N_PAR[case['model']]
    pts = float(n) * case['res'] * (0.525 if case.get('ragged') else 1.)
    tri = 2. * P * (P + 1)
    arms = _n_arms(case)
    if kind in ('snr', 'snr_call'):
        return {'bytes': 8. * n * (P + 1), 'flops': 4. * pts * arms}
    if kind in ('fisher', 'fisher_call', 'fisher_duty'):
        return {'bytes': 8. * n * (P + P * P), 'flops': tri * pts * arms}
    if kind == 'fisher_arms':
        return {'bytes': 8. * n * (P + arms * P * P), 'flops': tri * pts * arms}
    if kind == 'strain_grad':  # grid and gradient in, strain out; the Jacobian need not exist
        return {'bytes': 8. * (pts * (1 + 2 + 2) + 2. * n * P), 'flops': 4. * pts * P}
    return {'bytes': 8. * (pts * (2 + 2 + 2 * P) + n * (P + P * P)), 'flops': tri * pts}


# ------------------------------------------------------- values in 64 bits
def _psd_interp(path, f):
    t = np.loadtxt(path, usecols=(0, 1))
    return torch.from_numpy(np.interp(f.numpy(), t[:, 0], t[:, 1] ** 2, left=1., right=1.))


def _tf2_signal(x, f, site, rot, motion):
    """(Ap, Ac, Psi) of the TaylorF2 strain, 3.5PN with spins and tides, of
    the parameter rows x (P, N) on the grid f (N_f, N); plain torch."""
    pi = math.pi
    Mc, eta, dL, theta, phi, iota, psi, tc, Phic, c1, c2 = x[:11]
    T = glob.GMsun_over_c3
    M = Mc * T / eta ** 0.6
    v = (pi * M * f) ** (1. / 3.)
    lv = torch.log(v)
    e2, e3 = eta * eta, eta ** 3
    d = torch.sqrt(1. - 4. * eta)
    q1, q2 = 0.5 * (1. + d), 0.5 * (1. - d)
    s, a, ss, g = 0.5 * (c1 + c2), 0.5 * (c1 - c2), c1 * c2, np.euler_gamma
    p2 = 3715. / 756 + 55. / 9 * eta
    p3 = -16. * pi + 113. / 3 * d * a + (113. / 3 - 76. / 3 * eta) * s

    def quad(q, c):     # self-spin terms of one body, unit quadrupole
        return (-480. + 1. - 7.) / 9.6 * (q * c) ** 2

    p4 = (15293365. / 508032 + 27145. / 504 * eta + 3085. / 72 * e2 - 474. / 4.8 * eta * ss + quad(q1, c1) + quad(q2, c2))
    b5 = (38645. / 756 * pi - 65. / 9 * pi * eta - (732985. / 2268 - 24260. / 81 * eta - 340. / 9 * e2) * s
          - (732985. / 2268 + 140. / 9 * eta) * d * a)

    def spin6(q, c):
        return (pi * c * q * (1490. / 3 + 260. * q)
                + (4703.5 / 8.4 - 4108.25 / 6.72 + (2935. / 6 - 108.5 / 1.2) * q + (125.5 / 3.6 - 120.) * q * q) * (q * c) ** 2)

    p6 = (11583231236531. / 4694215680 - 640. / 3 * pi ** 2 - 6848. / 21 * g
          + eta * (-15737765635. / 3048192 + 2255. / 12 * pi ** 2) + 76055. / 1728 * e2 - 127825. / 1296 * e3
          - 6848. / 21 * math.log(4.) + spin6(q1, c1) + spin6(q2, c2) + (32675. / 112 + 5575. / 18 * eta) * eta * ss)
    p7 = (77096675. / 254016 * pi + 378515. / 1512 * pi * eta - 74045. / 756 * pi * e2
          + (-25150083775. / 3048192 + 10566655595. / 762048 * eta - 1042165. / 3024 * e2 + 5345. / 36 * e3) * s
          + d * (-25150083775. / 3048192 + 26804935. / 6048 * eta - 1985. / 48 * e2) * a)
    ph = (1. + p2 * v ** 2 + p3 * v ** 3 + p4 * v ** 4 + b5 * (1. + 3. * lv) * v ** 5 + (p6 - 6848. / 21 * lv) * v ** 6
          + p7 * v ** 7)
    if x.shape[0] > 11:
        ph = ph - 19.5 * x[11] * v ** 10 + (-3115. / 64 * x[11] + 6595. / 364 * d * x[12]) * v ** 12
    phase = 3. / (128. * eta) * ph / v ** 5 + 0.75 * pi
    amp = math.sqrt(5. / 24) * pi ** (-2. / 3) * glob.clightGpc / dL * (T * Mc) ** (5. / 6) * f ** (-7. / 6)
    t = tc + 0. * f
    if motion:
        tau = 5. / 256 * M / (eta * v ** 8) * (
            1. + (743. / 252 + 11. / 3 * eta) * v ** 2 - 32. / 5 * pi * v ** 3
            + (3058673. / 508032 + 5429. / 504 * eta + 617. / 72 * e2) * v ** 4 - (7729. / 252 - 13. / 3 * eta) * pi * v ** 5
            + (-10052469856691. / 23471078400 + 128. / 3 * pi ** 2 + 6848. / 105 * g
               + (3147553127. / 3048192 - 451. / 12 * pi ** 2) * eta - 15211. / 1728 * e2 + 25565. / 1296 * e3
               + 3424. / 105 * torch.log(16. * v * v)) * v ** 6
            + (-15419335. / 127008 - 75703. / 756 * eta + 14809. / 378 * e2) * pi * v ** 7)
        t = tc - tau / 86400.
    lat, lon = math.radians(site['lat']), math.radians(site['long'])
    xi = 2. * (math.radians(site['xax']) + math.radians(rot))
    dec = 0.5 * pi - theta
    delay = -glob.REarth / glob.clight * (torch.cos(dec) * math.cos(lat) * torch.cos(phi - lon - 2. * pi * t)
                                          + torch.sin(dec) * math.sin(lat))
    w = phi - lon - 2. * pi * (t + delay / 86400.)
    sx, cx, sl, cl = math.sin(xi), math.cos(xi), math.sin(lat), math.cos(lat)
    a_ = (sx / 16. * (3. - math.cos(2 * lat)) * (3. - torch.cos(2 * dec)) * torch.cos(2 * w)
          - 0.25 * cx * sl * (3. - torch.cos(2 * dec)) * torch.sin(2 * w)
          + 0.25 * sx * math.sin(2 * lat) * torch.sin(2 * dec) * torch.cos(w) - 0.5 * cx * cl * torch.sin(2 * dec) * torch.sin(w)
          + 0.75 * sx * (cl * torch.cos(dec)) ** 2)
    b_ = (cx * sl * torch.sin(dec) * torch.cos(2 * w) + 0.25 * sx * (3. - math.cos(2 * lat)) * torch.sin(dec) * torch.sin(2 * w)
          + cx * cl * torch.cos(dec) * torch.cos(w) + 0.5 * sx * math.sin(2 * lat) * torch.cos(dec) * torch.sin(w))
    z = 1. if site['shape'] == 'L' else math.sin(pi / 3)
    Fp = z * (a_ * torch.cos(2 * psi) + b_ * torch.sin(2 * psi))
    Fc = z * (b_ * torch.cos(2 * psi) - a_ * torch.sin(2 * psi))
    ci = torch.cos(iota)
    return (amp * Fp * 0.5 * (1. + ci * ci), amp * Fc * ci,
            2. * pi * f * tc * 86400. - Phic - phase + 2. * pi * f * delay)


def _tf2_rows(x, f, site, rot, motion):
    """Derivative rows without the common factor exp(i Psi): (P, N_f, N)."""
    rows = []
    for p in range(x.shape[0]):
        dx = torch.zeros_like(x)
        dx[p] = 1. / 86400. if p == 7 else 1.
        (Ap, Ac, Psi), (dp, dc, ds) = torch.func.jvp(lambda y: _tf2_signal(y, f, site, rot, motion), (x,), (dx,))
        rows.append(torch.complex(dp - Ac * ds, dc + Ap * ds))
    return torch.stack(rows), torch.complex(Ap, Ac), Psi


def _trapz_weights(f):
    w = torch.zeros_like(f)
    w[1:] += 0.5 * (f[1:] - f[:-1])
    w[:-1] += 0.5 * (f[1:] - f[:-1])
    return w


def _exact_tf2(case, seed):
    """TaylorF2 cases of up to 2 x 10^6 points x arms, else None."""
    if case['model'] not in ('TaylorF2', 'TaylorF2_tidal') or case['n'] * case['res'] * _n_arms(case) > 2e6:
        return None
    kind, motion = case['kind'], case['motion']
    ev, bns = _events(case, seed)
    x = torch.from_numpy(E.param_rows(ev, bns))
    n, P, res = x.shape[1], x.shape[0], case['res']
    if kind == 'strain_grad':
        f, wgt = (torch.from_numpy(a) for a in _misfit_inputs(case, seed))
    else:
        fcut = (1. / (6. * np.pi * np.sqrt(6.) * glob.GMsun_over_c3)) / (ev['Mc'] / ev['eta'] ** 0.6)
        if case.get('ragged'):
            return None
        f = torch.from_numpy(np.geomspace(np.full(n, 2.), fcut, res))
    arms = []
    for name, psd in NETS[case['net']]:
        site = glob.detectors[name]
        arms += [(site, 60. * k, PSD[psd]) for k in range(3 if site['shape'] == 'T' else 1)]
    w = _trapz_weights(f)
    if kind in ('snr', 'snr_call'):
        tot = 0.
        for site, rot, psd in arms:
            Ap, Ac, _ = _tf2_signal(x, f, site, rot, motion)
            tot = tot + ((Ap * Ap + Ac * Ac) / _psd_interp(psd, f) * w).sum(0)
        return 2. * torch.sqrt(tot)
    if kind == 'strain_grad':
        r, u, Psi = _tf2_rows(x, f, arms[0][0], 0., motion)
        e = torch.polar(torch.ones_like(Psi), Psi)
        r = r * e
        g = (wgt[None, ..., 0] * r.real + wgt[None, ..., 1] * r.imag).sum(1)
        g[7] *= 86400.
        return torch.view_as_real(u * e), g
    Fs = []
    masks = np.concatenate(_duty_masks(case, seed)) if kind == 'fisher_duty' else None
    for k, (site, rot, psd) in enumerate(arms[:1] if kind == 'derivatives' else arms):
        r, u, Psi = _tf2_rows(x, f, site, rot, motion)
        m = r * torch.sqrt(4. * w / _psd_interp(psd, f))
        m = torch.cat((m.real, m.imag), dim=1).permute(2, 0, 1)
        F = torch.matmul(m, m.transpose(1, 2)).permute(1, 2, 0)
        Fs.append(F if masks is None else F * torch.from_numpy(masks[k]))
    if kind == 'fisher_arms':
        return torch.stack(Fs)
    if kind == 'derivatives':
        e = torch.polar(torch.ones_like(Psi), Psi)
        return torch.view_as_real(u * e), torch.view_as_real((r * e).permute(0, 2, 1).contiguous()), Fs[0]
    return sum(Fs)


def _exact_screen(case, seed):
    """The network on its own bf16 weights, everything after them in 64 bits."""
    if case['n'] > 200000:
        return None
    ev, proxy = _screen_inputs(case, seed)
    dphi = ev['phi'] - 2. * np.pi * ev['tcoal']
    raw = np.stack([np.log(ev['Mc']), ev['eta'], np.log(ev['dL']), np.cos(ev['theta']), np.cos(dphi), np.sin(dphi),
                    np.cos(ev['iota']), np.cos(2 * ev['psi']), np.sin(2 * ev['psi']), ev['chi1z'], ev['chi2z']], axis=1)
    sd = raw.std(axis=0)
    x = torch.from_numpy((raw - raw.mean(axis=0)) / sd)
    par, o = {}, 0
    flat = screen.init_params(seed)
    for name, shape in screen.LAYOUT:
        k = int(np.prod(shape))
        t = torch.from_numpy(flat[o:o + k].reshape(shape))
        par[name] = (t.to(torch.bfloat16) if name in ('W1', 'W2', 'W3') else t).to(torch.float64)
        o += k
    par['W1'] = par['W1'][:, :x.shape[1]]
    for t in par.values():
        t.requires_grad_(case['kind'] == 'screen_step')
    h = x
    for l in '123':
        h = torch.nn.functional.silu(h @ par['W' + l].T + par['b' + l])
    y = h @ par['w4'] + par['b4']
    if case['kind'] == 'screen':
        return y.detach() * float(proxy.std()) + float(proxy.mean())
    target = torch.from_numpy((proxy - proxy.mean()) / proxy.std())
    grads = torch.autograd.grad(((y - target) ** 2).mean(), [par[name] for name, _ in screen.LAYOUT])
    out = []
    for (name, shape), g in zip(screen.LAYOUT, grads):
        full = torch.zeros(shape, dtype=torch.float64)
        if name == 'W1':
            full[:, :g.shape[1]] = g
        else:
            full = g
        out.append(full.reshape(-1))
    return y.detach(), torch.cat(out)


def exact(case, seed):
    """Plain 64-bit values; None for the IMRPhenomD models, whose 64-bit value
    is as long a program as the models themselves, and where plain
    arithmetic would take too long."""
    if case['kind'] in WAVE_KINDS:
        return _exact_tf2(case, seed)
    if case['kind'] in ('screen', 'screen_step'):
        return _exact_screen(case, seed)
    F = _fisher_batch(case, seed).transpose(2, 0, 1)
    s = 1. / np.sqrt(np.einsum('nii->ni', F))
    A = F * s[:, :, None] * s[:, None, :]
    C = np.linalg.inv(A)
    C = 0.5 * (C + C.transpose(0, 2, 1)) * s[:, :, None] * s[:, None, :]
    lam = np.linalg.eigvalsh(A)
    return np.ascontiguousarray(C.transpose(1, 2, 0)), np.abs(lam).max(axis=1) / np.abs(lam).min(axis=1), None
