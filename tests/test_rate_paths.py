"""Rate constants at the edges of their paths: every kind of reaction, layers
from one workgroup to eight layers per workgroup, temperatures either side of
the polynomials' break at 1000 K and far out of it, exponents beyond the range
that is formed in two doubles, powers of CORR T other than -1, 0 and 1.

Tolerance: both sides evaluate the same expressions; an exponent of up to 650
carries half an ulp (7e-14), so 1e-12 covers it, log and pow of each side and
the few products behind them.  Rates outside [1e-290, 1e290] only have to be
outside on both sides (zero, infinite and NaN alike)."""
import ctypes as C

import numpy as np
import pytest

from oracle import ros2_oracle as O
from vulcan_amd import _lib
from vulcan_amd import network as nw
from vulcan_amd import workloads as W

gpu = pytest.mark.gpu
TOL = 1e-12


def _network():
    net = W.full_network()
    rng = np.random.default_rng(5)
    kind, par = net.kind.copy(), net.par.copy()
    troe = np.flatnonzero(kind == nw.KIND_TROE)
    kind[troe[0::4]] = nw.KIND_LIND
    kind[troe[1::4]] = nw.KIND_K0
    kind[troe[2]] = nw.KIND_CH3OH
    arrh = np.flatnonzero(kind == nw.KIND_ARRH)
    par[arrh[0::7], nw.P_N] = rng.uniform(-10, 10, len(arrh[0::7]))
    par[arrh[1::7], nw.P_E] = rng.uniform(-2e4, 2e5, len(arrh[1::7]))
    par[arrh[2::7], nw.P_A] = 0.0
    par[arrh[3::7], nw.P_N] = 0.0
    reac, prod = net.reac.copy(), net.prod.copy()
    reac[arrh[4::14], 3] = 3            # one more reactant, one more product: other powers of CORR T
    reac[arrh[4::28], 2] = 5
    prod[arrh[5::14], 2:] = (7, 9)
    import dataclasses
    return dataclasses.replace(net, kind=kind, par=par, reac=reac, prod=prod)


@gpu
@pytest.mark.parametrize('layers', [2, 150, 4099, 8195, 16391])
@pytest.mark.parametrize('tau', [False, True])
def test_rates_of_every_path(layers, tau):
    import torch
    if not torch.cuda.is_available():
        pytest.skip('no HIP device')
    from vulcan_amd.device import DeviceColumns, DevicePlan, dptr, stream_handle
    net = _network()
    rng = np.random.default_rng(layers)
    some = np.array([1000.0, np.nextafter(1000.0, 0), 999.0, 60.0, 200.0, 6000.0, 3.0, 2e4, 1e-310, 0.0])
    T = rng.uniform(300, 3000, layers)
    T[:min(layers, len(some))] = some[:layers]
    T = rng.permutation(T)
    M, ta = 10.0 ** rng.uniform(8, 20, layers), 10.0 ** rng.uniform(-4, 2, layers)
    d = [torch.as_tensor(a, device='cuda') for a in (T, M, ta)]
    k = torch.full((layers, net.nr), -1.0, dtype=torch.float64, device='cuda')
    plan, cols = DevicePlan(net), DeviceColumns([layers])
    atm = _lib.Atm(Tco=dptr(d[0]), M=dptr(d[1]), **(dict(tau=dptr(d[2])) if tau else {}))
    _lib.check(_lib.load().vk_rates(plan.handle, cols.handle, C.byref(atm), dptr(k), stream_handle()), 'vk_rates')
    k = k.cpu().numpy()
    pick = np.unique(np.concatenate([np.flatnonzero(np.isin(T, some)), rng.integers(0, layers, 200), [0, layers - 1]]))
    with np.errstate(all='ignore'):
        ref = O.rates(net, T[pick], M[pick], ta[pick] if tau else None)
    k = k[pick]
    mid = (np.abs(ref) > 1e-290) & (np.abs(ref) < 1e290)
    assert mid.mean() > 0.5
    assert (np.abs(k[mid] - ref[mid]) <= TOL * np.abs(ref[mid])).all()
    assert np.array_equal(np.isnan(k), np.isnan(ref))
    assert (np.abs(k[np.abs(ref) <= 1e-290]) <= 1.1e-290).all()
    assert (np.abs(k[np.abs(ref) >= 1e290]) >= 0.9e290).all()
