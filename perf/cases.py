"""Timed cases of the framework's main paths, through its public entry points.

Seven kinds of work, each what a user's program does over and over:

* ``steps``    Ros2 attempts of a batch of columns of one network
               (``ColumnBatch.integrate``), from one column to hundreds;
* ``mixed``    the same over several networks at once (``MixedBatch``);
* ``solve``    one factorisation and refined solve of the block-tridiagonal
               Ros2 system (``vk_block_solve_system`` of the C ABI);
* ``rates``    the rate constants of a batch (``ColumnBatch.compute_rates``);
* ``photo``    one radiative-transfer update of the photolysis rates
               (``DevicePhoto.update``);
* ``predict``  forward pass of the warm-start network (``MLP.forward``);
* ``train``    one training step of it (``loss_and_backward``, ``adam_step``).

Column inputs follow the seeded workloads of ``vulcan_amd.workloads``:
isothermal-plus-gradient temperature with top and bottom uniform on
[400, 2500] K, Kzz log-uniform on [1e5, 1e11] cm2/s, pressure 1e3 to 1e-2
bar, a start near chemical equilibrium, dt0 = 1e-10 s, all in FP64.
"""
import ctypes as C
import functools
import math

import numpy as np
import torch

from vulcan_amd import _lib
from vulcan_amd import network as nw
from vulcan_amd import photo as P
from vulcan_amd.atmosphere import build_column
from vulcan_amd.config import Config
from vulcan_amd.device import ColumnBatch, DeviceColumns, DevicePlan, MixedBatch, dptr, stream_handle
from vulcan_amd.equilibrium import equilibrium
from vulcan_amd.mlp import MLP
from vulcan_amd.workloads import ColumnCase, element_vector, iso_gradient_profile

P_BOT, P_TOP = 1e9, 1e4                  # dyn/cm2
MLP_NZ = 150                             # layers of the warm-start network's columns
MLP_IN, MLP_HIDDEN = 2 * MLP_NZ + 7, 1024
GRP = 93                                 # species of the full-size network


def listed():
    return [
        # interactive use and quick tests: the small network on one column, where launches and latency decide
        dict(name='steps_small', kind='steps', ni=30, pairs=150, ncols=1, nz_lo=60, nz_hi=60, attempts=20, graph=True),
        # the plain method at full size: one column of 93 species, 600 reactions and 20 photolysis channels
        dict(name='steps_column', kind='steps', ni=93, pairs=620, ncols=1, nz_lo=150, nz_hi=150, attempts=10,
             graph=True),
        # a handful of ragged columns on the way to steady state: history kept, conv() evaluated, eager launches
        # (as the steady-state runs drive the loop)
        dict(name='steps_few', kind='steps', ni=93, pairs=620, ncols=12, nz_lo=80, nz_hi=200, attempts=4, graph=False,
             history=True),
        # an odd network with the transport and boundary options on: upwind vz and vm operators, top and bottom
        # fluxes with deposition, diffusion-limited escape
        dict(name='steps_options', kind='steps', ni=61, pairs=415, ncols=3, nz_lo=51, nz_hi=97, attempts=6, graph=True,
             options=True),
        # a grid of models: 256 uneven columns sharing the full-size network
        dict(name='steps_batch', kind='steps', ni=93, pairs=620, ncols=256, nz_lo=80, nz_hi=200, attempts=2,
             graph=True),
        # several chemistries at once: 40, 93 and 150 species, each network's columns on its own stream
        dict(name='steps_mixed', kind='mixed', ncols=240, nz_lo=100, nz_hi=150, attempts=1),
        # the linear solver alone, for a program with its own assembly (150 species, the largest network)
        dict(name='solve_blocks', kind='solve', ni=150, ncols=9, nz_lo=61, nz_hi=110, refine=1),
        # rate constants after a change of the temperature profiles of a batch
        dict(name='rates_batch', kind='rates', ni=93, pairs=620, ncols=256, nz_lo=80, nz_hi=200),
        # photolysis refresh of one column, as the loop of a photochemical run makes it
        dict(name='photo_column', kind='photo', ni=93, pairs=620, ncols=1, nz_lo=150, nz_hi=150, nbin=2588),
        # and of a batch of ragged columns
        dict(name='photo_batch', kind='photo', ni=93, pairs=620, ncols=48, nz_lo=80, nz_hi=200, nbin=2588),
        # warm-start prediction for a chunk of columns
        dict(name='predict', kind='predict', rows=256, hidden=MLP_HIDDEN, layers=4),
        # one minibatch of the warm-start network's training
        dict(name='train', kind='train', rows=256, hidden=MLP_HIDDEN, layers=4),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(['steps', 'steps', 'steps', 'steps', 'mixed', 'solve', 'rates', 'photo', 'predict', 'train'])
    if kind in ('predict', 'train'):
        return dict(kind=kind, rows=_log_int(rng, 8, 256), hidden=rng.choice([256, 500, 1024]), layers=rng.randint(2, 4))
    nz_lo = rng.randint(40, 150)
    nz_hi = rng.randint(nz_lo, min(200, nz_lo + 90))
    if kind == 'mixed':
        return dict(kind=kind, ncols=_log_int(rng, 6, 200), nz_lo=min(nz_lo, 120), nz_hi=min(nz_hi, 140), attempts=1)
    ni = rng.randint(27, 150)
    pairs = 150 if ni < 33 else 6 * ni + rng.randint(0, ni // 2)
    if kind == 'solve':
        return dict(kind=kind, ni=ni, ncols=_log_int(rng, 1, 9), nz_lo=min(nz_lo, 80), nz_hi=min(nz_hi, 100),
                    refine=rng.randint(0, 2))
    if kind == 'rates':
        return dict(kind=kind, ni=ni, pairs=pairs, ncols=_log_int(rng, 1, 160), nz_lo=nz_lo, nz_hi=nz_hi)
    if kind == 'photo':
        return dict(kind=kind, ni=ni, pairs=pairs, ncols=_log_int(rng, 1, 40), nz_lo=nz_lo, nz_hi=nz_hi,
                    nbin=rng.randint(700, 2588))
    # at most the work of steps_batch
    room = 256 * 140 * 93 ** 3 // (nz_hi * ni ** 3)
    ncols = _log_int(rng, 1, max(1, min(256, room)))
    attempts = rng.randint(2, max(2, min(10, 2 * room // ncols)))
    return dict(kind='steps', ni=ni, pairs=pairs, ncols=ncols, nz_lo=nz_lo, nz_hi=nz_hi, attempts=attempts,
                graph=rng.random() < 0.7, options=rng.random() < 0.25, history=rng.random() < 0.25)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

@functools.lru_cache(maxsize=None)
def _network(ni, pairs):
    """The seeded network of a size: 15 % of the pairs termolecular and 20
    photolysis channels from 600 pairs on, bimolecular alone below."""
    photo = 20 if pairs >= 600 else 0
    tb = (pairs - photo) * 15 // 100 if ni >= 60 else 0
    return nw.synthetic_network(ni, pairs - photo - tb, tb, photo, seed=1001 + ni, extra_elements=3 if ni > 110 else 0)


def _mixed_networks():
    return [_network(40, 200), _network(93, 620), _network(150, 1100)]


@functools.lru_cache(maxsize=None)
def _equilibrium_table(ni, pairs):
    """log mole fractions at equilibrium on a (T, log P) grid, from which the starts are interpolated."""
    net = _network(ni, pairs)
    T, lp = np.linspace(390., 2510., 20), np.linspace(np.log10(P_TOP), np.log10(P_BOT), 12)
    TT, LL = np.meshgrid(T, lp, indexing='ij')
    x = equilibrium(net, TT.ravel(), 10.0 ** LL.ravel(), element_vector(net))
    return T, lp, np.log(np.maximum(x, 1e-30)).reshape(len(T), len(lp), ni)


def _start_mix(ni, pairs, Tco, nz):
    T, lp, tab = _equilibrium_table(ni, pairs)
    u = np.clip((Tco - T[0]) / (T[1] - T[0]), 0, len(T) - 1.001)
    v = np.clip((np.linspace(lp[-1], lp[0], nz) - lp[0]) / (lp[1] - lp[0]), 0, len(lp) - 1.001)
    i, j = u.astype(int), v.astype(int)
    a, b = (u - i)[:, None], (v - j)[:, None]
    x = np.exp((1 - a) * ((1 - b) * tab[i, j] + b * tab[i, j + 1]) + a * ((1 - b) * tab[i + 1, j] + b * tab[i + 1, j + 1]))
    return x / x.sum(axis=1, keepdims=True)


def _layers(case, ncols):
    """Layer counts of a case's columns: uniform on its range, the same for every seed."""
    return [int(n) for n in np.random.default_rng([ncols, 11]).integers(case['nz_lo'], case['nz_hi'] + 1, ncols)]


def _columns(ni, pairs, case, seed, ncols, cfg):
    net = _network(ni, pairs)
    out = []
    for s, nz in zip(np.random.SeedSequence([seed, ni]).spawn(ncols), _layers(case, ncols)):
        rng = np.random.default_rng(s)
        T_top, T_bot = rng.uniform(400., 2500., 2)
        prof = iso_gradient_profile(nz, T_top, T_bot, P_BOT, P_TOP)
        x = _start_mix(ni, pairs, prof, nz)
        col = build_column(net, nz, T_bot, T_top, P_b=P_BOT, P_t=P_TOP, Kzz_bot=10.0 ** rng.uniform(5, 11), ymix0=x,
                           cfg=cfg, tau_top=1e-4, tau_bot=1e2, T_profile=prof)
        if case.get('options'):
            col.vz = rng.uniform(-5., 5., nz - 1)
            col.top_flux = -rng.uniform(0., 1e7, ni)
            col.bot_flux = rng.uniform(0., 1e7, ni)
            col.bot_vdep = rng.uniform(0., 1e-2, ni)
        out.append(ColumnCase(net=net, col=col, y0=col.M[:, None] * x, cfg=cfg))
    return net, out


def _config(case):
    if case.get('options'):
        return Config(use_vm_mol=True, use_vz=True, use_topflux=True, use_botflux=True, diff_esc=['H'])
    return Config()


# what an integration changes (state and, every update_frq steps, the geometry)
EVOLVES = ('y', 'ymix', 'y_prev', 'atom_loss', 'atom_loss_prev', 'state', 'mu', 'g', 'Hp', 'dz', 'zco', 'dzi', 'Hpi',
           'top_flux')


def _checkpoint(b):
    return [(getattr(b, n), getattr(b, n).clone()) for n in EVOLVES if getattr(b, n) is not None]


def _restore(saved):
    for now, then in saved:
        now.copy_(then)


def _step_outputs(b):
    """The composition and the step control's results.  delta, the clipped sums and the element losses are left
    out: near equilibrium they are differences at the last bits of the state."""
    f = b.state.view(torch.float64).view(-1, 12)
    i = b.state.view(torch.int32).view(-1, 24)
    return dict(y=b.y, ymix=b.ymix, t=f[:, 0], dt=f[:, 1], counters=i[:, 16:])


def _photo_tables(case, net, layout, seed):
    """Radiative-transfer tables with the shapes and magnitudes of a C-H-O network's: 0.1 nm bins to 240 nm and
    2 nm bins above, 17 absorbers with thresholds, two of them with a temperature dependence, H2 and He scattering,
    36 branches."""
    rng = np.random.default_rng([seed, 7])
    nb = case['nbin']
    n2 = nb // 12
    bins = np.concatenate([240. - 0.1 * np.arange(nb - n2, 0, -1), 240. + 2. * np.arange(n2)])
    nabs, nbr = 17, 36
    species = [int(s) for s in rng.choice(net.ni - 1, nabs, replace=False)]
    edge = rng.uniform(150., 400., nabs)[:, None]
    peak = 10.0 ** rng.uniform(-16.8, -15.4, nabs)[:, None]
    cross = peak * np.exp(-((bins - rng.uniform(60., 160., nabs)[:, None]) / rng.uniform(30., 90., nabs)[:, None]) ** 2)
    cross = np.where(bins < edge, cross, 0.0)
    br_abs = np.concatenate([np.arange(nabs), rng.integers(0, nabs, nbr - nabs)])
    cross_J = cross[br_abs] * rng.uniform(0.1, 1.0, nbr)[:, None]
    abs_T = [0, 1] + [-1] * (nabs - 2)
    TJ = [q for q in range(nbr) if br_abs[q] < 2]
    br_T = [TJ.index(q) if q in TJ else -1 for q in range(nbr)]
    f = rng.uniform(0.7, 1.3, (layout.L, 1))
    cross_T = np.stack([cross[a] * f for a in range(2)])
    cross_J_T = np.stack([cross_J[q] * f for q in TJ])
    scat = [net.species.index('H2'), net.species.index('He')]
    cross_scat = np.stack([8e-15 / bins ** 4 * 1e3, 5e-16 / bins ** 4 * 1e3])
    sflux = 10.0 ** (1.0 + 4.0 * np.clip((bins - 150.) / 300., 0, 1)) * rng.uniform(0.5, 1.5, nb)
    col = [int(c) for c in 2 * rng.choice(net.npairs, nbr, replace=False)]
    return P.PhotoTables(bins=bins, din12=nb - n2, sflux_top=sflux, abs_sp=species, abs_T=abs_T, cross=cross,
                         cross_T=cross_T, scat_sp=scat, cross_scat=cross_scat, br_col=col, br_T=br_T, cross_J=cross_J,
                         cross_J_T=cross_J_T, dbin1=0.1, dbin2=2., cos_sl=float(np.cos(48 / 180. * 3.14159)), edd=0.5,
                         f_diurnal=1., flux_atol=1.)


def _blocks(case, seed):
    """Block-tridiagonal systems shaped like the Ros2 lhs: c0 I - J - diffusion in units of c0, J with losses on the
    diagonal balanced by sparse productions over many decades, species scaled apart by orders of magnitude."""
    rng = np.random.default_rng([seed, 3])
    ni = case['ni']
    nz = _layers(case, case['ncols'])
    L = sum(nz)
    prod = 10.0 ** rng.uniform(-6, 3, (L, ni, ni)) * (rng.random((L, ni, ni)) < 0.3)
    lo, up = 10.0 ** rng.uniform(-4, 1, (L, ni)), 10.0 ** rng.uniform(-4, 1, (L, ni))
    d = np.arange(ni)
    prod[:, d, d] = 0.0
    D = -prod
    D[:, d, d] = 1.0 + prod.sum(axis=1) + lo + up
    s = 10.0 ** rng.uniform(-2, 2, ni)
    D *= s[:, None] / s
    off = np.concatenate([[0], np.cumsum(nz)])
    Lsub, Usup = -lo, -up
    Lsub[off[:-1]] = 0.0
    Usup[off[1:] - 1] = 0.0
    b = s * rng.standard_normal((L, ni))
    return nz, D, Lsub, Usup, b


def _mlp_data(case, seed):
    rng = np.random.default_rng([seed, 5])
    sizes = [MLP_IN] + [case['hidden']] * case['layers'] + [GRP * MLP_NZ]
    X = rng.standard_normal((case['rows'], sizes[0])).astype(np.float32)
    T = rng.standard_normal((case['rows'], sizes[-1])).astype(np.float32)
    return sizes, X, T


def prepare(case, seed):
    kind = case['kind']
    if kind in ('steps', 'rates'):
        cfg = _config(case)
        net, cases = _columns(case['ni'], case['pairs'], case, seed, case['ncols'], cfg)
        hist = cfg.conv_step + 1 if case.get('history') else 0
        b = ColumnBatch(DevicePlan(net), [c.col for c in cases], [c.y0 for c in cases], cfg, history=hist,
                        graph=bool(case.get('graph')), tune=kind == 'steps')
        return dict(kind=kind, batch=b, attempts=case.get('attempts'), saved=_checkpoint(b))
    if kind == 'mixed':
        cases = []
        for q, net in enumerate(_mixed_networks()):
            n = (case['ncols'] + 2 - q) // 3
            cases += _columns(net.ni, net.npairs, case, seed, n, Config())[1]
        mb = MixedBatch(cases)
        torch.cuda.synchronize()
        return dict(kind=kind, batch=mb, attempts=case['attempts'], saved=[_checkpoint(b) for _, b, _ in mb.groups])
    if kind == 'solve':
        nz, *arrays = _blocks(case, seed)
        plan, cols = DevicePlan(_network(case['ni'], 150 if case['ni'] < 33 else 6 * case['ni'])), DeviceColumns(nz)
        ms = (C.c_float * 5)()
        _lib.check(_lib.load().vk_tune_factor(plan.handle, cols.handle, 2, ms, stream_handle()), 'vk_tune_factor')
        D, Lsub, Usup, b = (torch.as_tensor(a, device='cuda') for a in arrays)
        return dict(kind=kind, plan=plan, cols=cols, D=D, Lsub=Lsub, Usup=Usup, b=b, x=torch.empty_like(b),
                    info=torch.zeros(case['ncols'], dtype=torch.int32, device='cuda'), refine=case['refine'])
    if kind == 'photo':
        net, cases = _columns(case['ni'], case['pairs'], case, seed, case['ncols'], Config())
        b = ColumnBatch(DevicePlan(net), [c.col for c in cases], [c.y0 for c in cases], Config(), tune=False)
        ph = P.DevicePhoto(b.plan, b.layout, _photo_tables(case, net, b.layout, seed))
        return dict(kind=kind, batch=b, photo=ph)
    sizes, X, T = _mlp_data(case, seed)
    return dict(kind=kind, mlp=MLP(sizes, seed=seed), X=torch.as_tensor(X, device='cuda'),
                T=torch.as_tensor(T, device='cuda'))


def run(state):
    kind = state['kind']
    if kind == 'steps':
        b = state['batch']
        _restore(state['saved'])
        b.integrate(state['attempts'])
        return _step_outputs(b)
    if kind == 'mixed':
        mb = state['batch']
        for (_, _, stream), saved in zip(mb.groups, state['saved']):
            with torch.cuda.stream(stream):
                _restore(saved)
        mb.integrate(state['attempts'])
        return [_step_outputs(b) for _, b, _ in mb.groups]
    if kind == 'solve':
        s = state
        _lib.check(_lib.load().vk_block_solve_system(s['plan'].handle, s['cols'].handle, dptr(s['D']), dptr(s['Lsub']),
                                                     dptr(s['Usup']), dptr(s['b']), dptr(s['x']), s['refine'],
                                                     dptr(s['info']), stream_handle()), 'vk_block_solve_system')
        return dict(x=s['x'], info=s['info'])
    if kind == 'rates':
        state['batch'].compute_rates()
        return state['batch'].k
    if kind == 'photo':
        b = state['batch']
        state['photo'].update(b.y, b.ymix, b.dz, b.k, state=b.state)
        return dict(k=b.k, change=b.state.view(torch.float64).view(-1, 12)[:, 7])
    mlp = state['mlp']
    if kind == 'predict':
        return mlp.forward(state['X'])
    loss, Y = mlp.loss_and_backward(state['X'], state['T'])
    mlp.adam_step(lr=1e-3, wd=1e-5)
    return dict(loss=loss, Y=Y, grads=mlp.grads, W=mlp.W, b=mlp.b, m=mlp.m, v=mlp.v,
                Wb=[w.view(torch.bfloat16) for w in mlp.Wb])


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------

def _step_work(ni, pairs, layers, attempts):
    """Per attempt: the blocks' elimination (8/3 ni^3 a layer), four solves and two residuals with the blocks (each
    two multiply-adds an entry), the rate products; per pass the state, the rates and the atmosphere once in, the
    state once out."""
    flops = layers * (8. / 3. * ni ** 3 + 4 * 4 * ni ** 2 + 2 * 2 * ni ** 2 + 3 * 10 * pairs)
    return 8. * layers * (2 * pairs + 4 * ni + 12), attempts * flops


def work(case):
    kind = case['kind']
    if kind in ('predict', 'train'):
        sizes = [MLP_IN] + [case['hidden']] * case['layers'] + [GRP * MLP_NZ]
        W = sum(a * b for a, b in zip(sizes, sizes[1:]))
        B = case['rows']
        if kind == 'predict':
            return dict(bytes=2. * W + 4. * sum(sizes[1:]) + 4. * B * (sizes[0] + sizes[-1]), flops=2. * B * W)
        # weights and moments in and out, the gradients and the BF16 copies out
        first = 2. * B * sizes[0] * sizes[1]
        return dict(bytes=(6 * 4. + 4. + 2.) * W + 4. * B * (sizes[0] + 2 * sizes[-1]), flops=3 * 2. * B * W - first)
    layers = case['ncols'] * (case['nz_lo'] + case['nz_hi']) / 2.
    if kind == 'mixed':
        parts = [_step_work(n.ni, n.npairs, layers / 3., case['attempts']) for n in _mixed_networks()]
        return dict(bytes=sum(p[0] for p in parts), flops=sum(p[1] for p in parts))
    ni = case['ni']
    if kind == 'solve':
        r = case['refine']
        return dict(bytes=8. * layers * (ni * ni + 4 * ni), flops=layers * (8. / 3. * ni ** 3 + (r + 1) * 4 * ni ** 2 + r * 2 * ni ** 2))
    if kind == 'rates':
        # a pair: about two pow and three exp or log of some 40 operations each
        return dict(bytes=8. * layers * (2 * case['pairs'] + 3), flops=layers * (200. * case['pairs'] + 120. * ni))
    if kind == 'photo':
        # per layer and bin: 19 absorbers and scatterers, about five exp or sqrt in the sweeps; 36 branches
        nb = case['nbin']
        return dict(bytes=8. * (layers * (2 * ni + 36) + nb * (17 + 2 + 36) + layers * nb * 4),
                    flops=layers * nb * (19 * 4. + 250. + 36 * 2.))
    b, f = _step_work(ni, case['pairs'], layers, case['attempts'])
    return dict(bytes=b, flops=f)


# ---------------------------------------------------------------------------
# 64-bit values
# ---------------------------------------------------------------------------

def _exact_rates(net, cols):
    out = []
    for c in cols:
        T, M, tau = c.col.Tco[:, None], c.col.M[:, None], c.col.tau[:, None]
        A, n, E, Ai, ni_, Ei, Fc, J0 = (net.par[None, :, q] for q in range(8))
        k0 = A * T ** n * np.exp(-E / T)
        with np.errstate(divide='ignore', invalid='ignore'):
            kinf = Ai * T ** ni_ * np.exp(-Ei / T)
            ff = np.exp(np.log(Fc) / (1. + (np.log(k0 * M / kinf) / (0.75 - 1.27 * np.log(Fc))) ** 2))
            troe = k0 / (1 + k0 * M / kinf) * ff
        kf = np.where(net.kind == nw.KIND_TROE, troe, np.where(net.kind == nw.KIND_PHOTO, J0 * np.exp(-tau), k0))
        a = [np.where(T < 1000, net.nasa9[None, :, q], net.nasa9[None, :, 10 + q]) for q in range(10)]
        h = (-a[0] / T ** 2 + a[1] * np.log(T) / T + a[2] + a[3] * T / 2 + a[4] * T ** 2 / 3 + a[5] * T ** 3 / 4
             + a[6] * T ** 4 / 5 + a[8] / T)
        s = (-a[0] / T ** 2 / 2 - a[1] / T + a[2] * np.log(T) + a[3] * T + a[4] * T ** 2 / 2 + a[5] * T ** 3 / 3
             + a[6] * T ** 4 / 4 + a[9])
        g = np.concatenate([h - s, np.zeros((len(T), 2))], axis=1)      # empty terms read the zeros
        dg = g[:, net.prod].sum(axis=2) - g[:, net.reac].sum(axis=2)
        dn = (net.reac >= 0).sum(axis=1) - (net.prod >= 0).sum(axis=1)
        K = np.exp(-dg) * (1.38064852E-16 / 1.e6 * T) ** dn
        k = np.zeros((len(T), net.nr))
        k[:, 0::2] = kf
        k[:, 1::2] = np.where(net.rev > 0, kf / K, 0.0)
        out.append(k)
    return np.concatenate(out)


def _exact_photo(t, cols, k):
    """First update of the columns (no upward flux before it); fills the branches' columns of k."""
    nb, mu = len(t.bins), -t.cos_sl
    change = []
    l0 = 0
    for c in cols:
        y, dz, nz = c.y0, c.col.dz, len(c.col.dz)
        ymix = y / y.sum(axis=1, keepdims=True)
        tau, w = np.zeros((nz + 1, nb)), np.zeros((nz, nb))
        sig = t.cross_scat
        for j in range(nz - 1, -1, -1):
            cr = np.stack([t.cross_T[q, l0 + j] if q >= 0 else t.cross[a] for a, q in enumerate(t.abs_T)])
            tau[j] = tau[j + 1] + dz[j] * (y[j, t.abs_sp] @ cr + y[j, t.scat_sp] @ sig)
            ta, ts = ymix[j, t.abs_sp] @ t.cross, ymix[j, t.scat_sp] @ sig
            w[j] = np.minimum(ts / (ta + ts), 1. - 1.E-8)
        sf = t.sflux_top * np.exp(-tau / t.cos_sl)
        s1 = np.sqrt(1. - w)
        tran = np.exp(-s1 / t.edd * (tau[:-1] - tau[1:]))
        zp, zm = 0.5 * (1 + s1), 0.5 * (1 - s1)
        ll = -w / (1. / mu ** 2 - (1. - w) / t.edd ** 2)
        gp, gm = 0.5 * ll * (1. / t.edd + 1. / mu), 0.5 * ll * (1. / t.edd - 1. / mu)
        chi, xi, phi = zm ** 2 * tran ** 2 - zp ** 2, zp * zm * (1. - tran ** 2), (zm ** 2 - zp ** 2) * tran
        lo, hi = sf[:-1] * t.cos_sl, sf[1:] * t.cos_sl
        iu = phi * gp * lo - (xi * gm + chi * gp) * hi
        idn = phi * gm * hi - (chi * gm + xi * gp) * lo
        du, dd = np.zeros((nz + 1, nb)), np.zeros((nz + 1, nb))
        for j in range(nz - 1, -1, -1):
            dd[j] = (phi[j] * dd[j + 1] + idn[j] / mu) / chi[j]
        for j in range(nz):
            du[j + 1] = (phi[j] * du[j] - xi[j] * dd[j + 1] + iu[j] / mu) / chi[j]
        tot = 0.5 * (sf[:-1] + sf[1:]) + 0.5 * (du[:-1] + du[1:] + dd[1:] + dd[:-1]) / t.edd
        af = tot / (t.hc / t.bins)
        d = t.din12
        for q, colno in enumerate(t.br_col):
            f = af * (t.cross_J_T[t.br_T[q], l0:l0 + nz] if t.br_T[q] >= 0 else t.cross_J[q])
            k[l0:l0 + nz, colno] = t.f_diurnal * (
                (f[:, :d].sum(axis=1) - 0.5 * (f[:, 0] + f[:, d - 1])) * t.dbin1
                + (f[:, d:].sum(axis=1) - 0.5 * (f[:, d] + f[:, -1])) * t.dbin2)
        change.append(1.0 if np.any(af > t.flux_atol) else 0.0)
        l0 += nz
    return dict(k=k, change=np.array(change))


def _exact_solve(nz, D, Lsub, Usup, b, steps=3):
    """Block elimination in 64 bits, refined with residuals in extended precision."""
    x = np.zeros_like(b)
    l0 = 0
    for n in nz:
        sl = slice(l0, l0 + n)
        d, lo, up = D[sl], Lsub[sl], Usup[sl]
        inv = np.empty_like(d)
        for j in range(n):
            s = d[j] if j == 0 else d[j] - lo[j][:, None] * inv[j - 1] * up[j - 1]
            inv[j] = np.linalg.inv(s)
        de, loe, upe = (v.astype(np.longdouble) for v in (d, lo, up))
        xe, r = np.zeros((n, d.shape[1]), np.longdouble), b[sl].astype(np.longdouble)
        for _ in range(steps):
            z = np.empty_like(b[sl])
            for j in range(n):
                z[j] = inv[j] @ (r[j].astype(float) - (lo[j] * z[j - 1] if j else 0.0))
            for j in range(n - 2, -1, -1):
                z[j] -= inv[j] @ (up[j] * z[j + 1])
            xe += z
            r = b[sl].astype(np.longdouble) - (de * xe[:, None, :]).sum(axis=2)
            r[1:] -= loe[1:] * xe[:-1]
            r[:-1] -= upe[:-1] * xe[1:]
        x[sl] = xe.astype(float)
        l0 += n
    return x


def _exact_mlp(case, seed):
    sizes, X, T = _mlp_data(case, seed)
    rng = np.random.default_rng(seed)
    f64 = dict(dtype=torch.float64, device='cuda')
    W = []
    for fi, fo in zip(sizes[:-1], sizes[1:]):
        w = rng.standard_normal((fi, fo)).astype(np.float32) * np.float32(np.sqrt(2.0 / fi))
        W.append(torch.as_tensor(w, device='cuda').to(torch.float64).requires_grad_())
    b = [torch.zeros(fo, requires_grad=True, **f64) for fo in sizes[1:]]
    A = torch.as_tensor(X, **f64)
    for l in range(len(W)):
        A = A @ W[l] + b[l]
        if l < len(W) - 1:
            A = torch.nn.functional.silu(A)
    if case['kind'] == 'predict':
        return A.detach()
    loss = ((A - torch.as_tensor(T, **f64)) ** 2).mean()
    loss.backward()
    p, g = [w.detach() for w in W + b], [w.grad for w in W + b]
    m, v, new = [], [], []
    for q, (w, d) in enumerate(zip(p, g)):
        d = d + (1e-5 * w if q < len(W) else 0.0)
        m.append(0.1 * d)
        v.append(0.001 * d * d)
        new.append(w - 1e-3 * d / (d.abs() + 1e-8))
    n = len(W)
    # the first update of a bias that starts at zero is lr times its gradient's sign: no value to compare where the
    # gradient is at rounding level
    return dict(loss=float(loss), Y=A.detach(), grads=g, W=new[:n], b=[None] * n, m=m, v=v, Wb=new[:n])


def exact(case, seed):
    kind = case['kind']
    if kind in ('predict', 'train'):
        return _exact_mlp(case, seed)
    if kind == 'solve':
        nz, D, Lsub, Usup, b = _blocks(case, seed)
        return dict(x=_exact_solve(nz, D, Lsub, Usup, b), info=None)
    if kind in ('rates', 'photo'):
        net, cols = _columns(case['ni'], case['pairs'], case, seed, case['ncols'], Config())
        k = _exact_rates(net, cols)
        if kind == 'rates':
            return k
        layout = DeviceColumns([c.col.nz for c in cols])
        return _exact_photo(_photo_tables(case, net, layout, seed), cols, k)
    # an integration decides each step's acceptance and size from rounding-level differences: no closed value
    return None
