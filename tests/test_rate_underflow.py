"""Reverse rates of forward rates near and below the smallest normal number:
cold layers and high barriers take k_f to 1e-314, and k_r = k_f / K of an
exothermic reaction is an ordinary number again, as accurate as the k_f it is
formed from.  Likewise k_f from a pre-exponential factor as small.

Tolerance: both sides form the exponential of up to 600 (half an ulp of it is
6e-14); 1e-12 covers it and the few products behind."""
import ctypes as C

import numpy as np
import pytest

from vulcan_amd import _lib
from vulcan_amd import network as nw

gpu = pytest.mark.gpu
TOL = 1e-12


@gpu
@pytest.mark.parametrize('layers', [7, 1409, 2817, 5633, 40000])      # one, two, four and eight layers a workgroup
def test_rates_of_tiny_factors(layers):
    import torch
    if not torch.cuda.is_available():
        pytest.skip('no HIP device')
    from vulcan_amd.device import DeviceColumns, DevicePlan, dptr, stream_handle
    dg = np.array([0., 100., 300., 500., 600.])             # -ln K of the pairs
    n = len(dg)
    nasa9 = np.zeros((2 * n, 20))
    nasa9[1::2, 9] = nasa9[1::2, 19] = -dg                   # g/RT of the products
    par = np.zeros((2 * n, 8))
    par[:n, nw.P_A], par[:n, nw.P_E] = 1.0, 725.0 * 100.0    # k_f of 1e-307 to 5e-322 over the layers below
    par[n:, nw.P_A] = 3.7e-314 * np.linspace(1, 2, n)        # and from such factors, T^100
    par[n:, nw.P_N] = 100.0
    one = np.full((2 * n, 4), -2, np.int32)
    reac, prod = one.copy(), one.copy()
    reac[:, 0], prod[:, 0] = np.tile(2 * np.arange(n), 2), np.tile(2 * np.arange(n) + 1, 2)
    net = nw.Network(species=['s%d' % i for i in range(2 * n)], elements=['H'], compo=np.ones((2 * n, 1), np.int32),
                     mass=np.full(2 * n, 2.0), nasa9=nasa9, reac=reac, prod=prod, kind=np.zeros(2 * n, np.int32), par=par,
                     rev=np.concatenate([np.ones(n, np.int32), np.zeros(n, np.int32)]))
    T = np.random.default_rng(layers).uniform(98., 102.5, layers)
    d = [torch.as_tensor(a, device='cuda') for a in (T, np.full(layers, 1e15))]
    k = torch.full((layers, net.nr), -1.0, dtype=torch.float64, device='cuda')
    plan, cols = DevicePlan(net), DeviceColumns([layers])
    _lib.check(_lib.load().vk_rates(plan.handle, cols.handle, C.byref(_lib.Atm(Tco=dptr(d[0]), M=dptr(d[1]))), dptr(k),
                                    stream_handle()), 'vk_rates')
    k = k.cpu().numpy()
    kf, kr = k[:, :2 * n:2], k[:, 1:2 * n:2]
    assert (kf > 0).all() and (kf < 1e-300).any()
    ref = kf / np.exp(-dg)
    big = ref > 1e-290
    assert big[:, 2:].all()
    assert (np.abs(kr[big] - ref[big]) <= TOL * ref[big]).all()
    ref = par[n:, nw.P_A] * T[:, None] ** par[n:, nw.P_N]
    assert (np.abs(k[:, 2 * n::2] - ref) <= TOL * ref).all()
