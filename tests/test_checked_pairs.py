"""The bounds-checked build sees a species index just beyond the network in a
pair's reactants or products: the packed tables use the two numbers beyond the
species for M and for an empty slot, and such an index must not pass for them."""
import json
import os
import subprocess
import sys

import pytest

from vulcan_amd import _lib

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
gpu = pytest.mark.gpu

RUN = r'''
import ctypes as C, dataclasses, json, sys
sys.path.insert(0, %(root)r)
import torch
from vulcan_amd import _lib
_lib.LIB_PATH = _lib.CHECKED_LIB_PATH
from vulcan_amd import device, workloads as W
from vulcan_amd.network import build_tables
from vulcan_amd.device import DeviceColumns, DevicePlan, dptr, stream_handle
lib, net = _lib.load(), W.small_network()
good = build_tables(net)
device.build_tables = lambda _: good             # the derived tables of the valid network
out = {}
for name, side, term in [('valid', 'reac', None)] + [(s + '%%+d' %% d, s, d) for s in ('reac', 'prod') for d in (0, 1, 2, 300)] + \
        [('reac-3', 'reac', -3 - net.ni)]:
    tab = getattr(net, side).copy()
    if term is not None:
        tab[7, 0] = net.ni + term
    plan, cols = DevicePlan(dataclasses.replace(net, **{side: tab})), DeviceColumns([2])
    y, k = (torch.ones((2, n), dtype=torch.float64, device='cuda') for n in (net.ni, net.nr))
    M, f = torch.ones(2, dtype=torch.float64, device='cuda'), torch.empty_like(y)
    site = C.c_int(-1)
    assert lib.vk_debug_checks(C.byref(site), 1) == 0
    _lib.check(lib.vk_chemdf(plan.handle, cols.handle, dptr(y), dptr(M), dptr(k), dptr(f), stream_handle()), 'vk_chemdf')
    torch.cuda.synchronize()
    assert lib.vk_debug_checks(C.byref(site), 0) == 0
    out[name] = site.value
print(json.dumps(out))
'''


@gpu
@pytest.mark.timeout(200)
def test_species_beyond_the_network_are_seen():
    import torch
    if not torch.cuda.is_available():
        pytest.skip('no HIP device')
    p = subprocess.run([sys.executable, '-c', RUN % {'root': ROOT}], capture_output=True, text=True, timeout=150)
    assert p.returncode == 0, p.stdout[-2000:] + p.stderr[-4000:]
    sites = json.loads(p.stdout.strip().splitlines()[-1])
    print(sites)
    assert sites.pop('valid') == 0
    assert all(s > 0 for s in sites.values()), sites


@gpu
@pytest.mark.parametrize('which,columns', [('small', 1), ('large', 1), ('small', 110), ('large', 110)])
def test_pairs_with_repeated_species_and_third_bodies(which, columns):
    """chemdf of pairs with a species two or three times on a side and with M in
    front and behind, one and two layers a workgroup, against the oracle."""
    import numpy as np
    import torch
    if not torch.cuda.is_available():
        pytest.skip('no HIP device')
    from oracle import ros2_oracle as O
    from test_jac_layers import _network
    from vulcan_amd import workloads as W
    from vulcan_amd.config import Config
    from vulcan_amd.device import ColumnBatch, DevicePlan, dptr, stream_handle
    net = _network(which)
    c = W.small_case(nz=41, net=net)
    b = ColumnBatch(DevicePlan(net), [c.col] * columns, [c.y0] * columns, Config(), tune=False)
    f = torch.empty_like(b.y)
    _lib.check(_lib.load().vk_chemdf(b.plan.handle, b.layout.handle, dptr(b.y), dptr(b.M), dptr(b.k), dptr(f),
                                     stream_handle()), 'vk_chemdf')
    f, k = f.cpu().numpy(), b.k.cpu().numpy()
    b.close()
    ref = O.chemdf(net, c.y0, c.col.M, k[:41])
    for q in (0, columns - 1):
        assert np.array_equal(f[41 * q:41 * (q + 1)], ref)
