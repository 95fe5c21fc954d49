"""Jacobian and left-hand-side blocks of networks small, medium and large, at
the numbers of layers where their kernels change (one layer a workgroup up to
one a CU; two beyond; from six a CU on, those of up to 61 species on 256 threads
for two layers instead of 512), with blocks that held other numbers before:
every entry, the structural zeros among them, against the oracle bit for bit."""
import ctypes as C

import numpy as np
import pytest

from oracle import ros2_oracle as O
from vulcan_amd import _lib
from vulcan_amd import network as nw
from vulcan_amd import workloads as W
from vulcan_amd.config import Config

gpu = pytest.mark.gpu


@gpu
@pytest.mark.parametrize('layers,extra', [(1, 0), (1, 1), (6, -1), (6, 1)])
@pytest.mark.parametrize('ni,pairs', [(27, 100), (30, 150), (61, 415), (93, 620), (150, 1100)])
def test_every_entry_is_written(ni, pairs, layers, extra):
    import torch
    if not torch.cuda.is_available():
        pytest.skip('no HIP device')
    from vulcan_amd.device import ColumnBatch, DevicePlan, dptr, stream_handle
    net = W.small_network() if ni == 30 else nw.synthetic_network(ni, pairs, 0, 0, seed=ni,
                                                                  extra_elements=3 if ni > 110 else 0)
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    nz = 32
    n = layers * cus // nz
    cases = [W.small_case(nz=nz, net=net)] * (n - 1) + [W.small_case(nz=nz + layers * cus % nz + extra, net=net)]
    rng = np.random.default_rng(ni + layers + extra)
    y0 = [c.y0 * rng.uniform(0.5, 2.0, c.y0.shape) for c in cases]
    dt = 10.0 ** rng.uniform(-9, -3, n)
    b = ColumnBatch(DevicePlan(net), [c.col for c in cases], y0, Config(), tune=False)
    L = b.layout.L
    assert L == layers * cus + extra
    lib = _lib.load()
    J, D = (torch.full((L, ni, ni), np.nan, dtype=torch.float64, device='cuda') for _ in range(2))
    Ls, Us = (torch.full((L, ni), np.nan, dtype=torch.float64, device='cuda') for _ in range(2))
    _lib.check(lib.vk_jac(b.plan.handle, b.layout.handle, dptr(b.y), dptr(b.M), dptr(b.k), dptr(J), stream_handle()),
               'vk_jac')
    d = torch.as_tensor(dt, device='cuda')
    _lib.check(lib.vk_lhs(b.plan.handle, b.layout.handle, C.byref(b.atm), dptr(b.y), dptr(b.k), 1, dptr(d), dptr(D),
                          dptr(Ls), dptr(Us), stream_handle()), 'vk_lhs')
    J, D, Ls, Us, k = (t.cpu().numpy() for t in (J, D, Ls, Us, b.k))
    off = b.layout.off
    b.close()
    for i in (0, n - 1):
        s = slice(off[i], off[i + 1])
        ref = O.jac_blocks(net, y0[i], cases[i].col.M, k[s])
        assert np.array_equal(J[s], ref)
        for a, r in zip((D, Ls, Us), O.lhs_blocks(cases[i].col, y0[i], dt[i], ref, True)):
            assert np.array_equal(a[s], r)
