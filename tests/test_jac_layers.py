"""Right-hand sides, Jacobian and left-hand-side blocks with two layers per workgroup (many
layers) against one (few layers), bit for bit: an odd number of layers, columns
of different lengths and time steps whose ends fall inside a pair of layers,
and pairs of reactions with a species twice on one side, in either order, and
with M.  The blocks of few layers are compared with the oracle, bit for bit."""
import ctypes as C
import dataclasses

import numpy as np
import pytest

from oracle import ros2_oracle as O
from vulcan_amd import _lib
from vulcan_amd import workloads as W
from vulcan_amd.config import Config

gpu = pytest.mark.gpu


def _network(which):
    net = W.small_network() if which == 'small' else W.mixed_networks()[2]
    reac, prod = net.reac.copy(), net.prod.copy()
    reac[0] = (3, 3, -2, -2)
    reac[1] = (4, 5, 4, -1)
    prod[2] = (6, 7, 6, 6)
    prod[3] = (-1, 8, 9, -2)
    return dataclasses.replace(net, reac=reac, prod=prod)


@gpu
@pytest.mark.parametrize('which,nz', [('small', 61), ('large', 101)])
def test_two_layers_per_workgroup(which, nz):
    import torch
    if not torch.cuda.is_available():
        pytest.skip('no HIP device')
    from vulcan_amd.device import ColumnBatch, DevicePlan, dptr, stream_handle
    net = _network(which)
    lib = _lib.load()
    one = W.small_case(nz=nz, net=net)
    two = W.small_case(nz=nz - 2, net=net)
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    n = (12 * cus) // nz + 3
    n += (n * nz + (nz - 2)) % 2 == 0            # an odd number of layers
    cases = [one] * n + [two]
    rng = np.random.default_rng(3)
    y0 = [c.y0 * rng.uniform(0.5, 2.0, c.y0.shape) for c in cases]
    dt = 10.0 ** rng.uniform(-9, -3, len(cases))

    def blocks(sel, mol):
        b = ColumnBatch(DevicePlan(net), [cases[i].col for i in sel], [y0[i] for i in sel], Config(), tune=False)
        L, ni = b.y.shape
        J, D = (torch.full((L, ni, ni), np.nan, dtype=torch.float64, device='cuda') for _ in range(2))
        Ls, Us = (torch.full((L, ni), np.nan, dtype=torch.float64, device='cuda') for _ in range(2))
        d = torch.as_tensor(dt[sel], device='cuda')
        _lib.check(lib.vk_jac(b.plan.handle, b.layout.handle, dptr(b.y), dptr(b.M), dptr(b.k), dptr(J),
                              stream_handle()), 'vk_jac')
        _lib.check(lib.vk_lhs(b.plan.handle, b.layout.handle, C.byref(b.atm), dptr(b.y), dptr(b.k), mol, dptr(d),
                              dptr(D), dptr(Ls), dptr(Us), stream_handle()), 'vk_lhs')
        f, g = torch.empty_like(b.y), torch.empty_like(b.y)
        _lib.check(lib.vk_chemdf(b.plan.handle, b.layout.handle, dptr(b.y), dptr(b.M), dptr(b.k), dptr(f),
                                 stream_handle()), 'vk_chemdf')
        _lib.check(lib.vk_diffdf(b.plan.handle, b.layout.handle, C.byref(b.atm), dptr(b.y), mol, dptr(g),
                                 stream_handle()), 'vk_diffdf')
        out = [t.cpu().numpy() for t in (J, D, Ls, Us, f, g, b.k)]
        b.close()
        return out

    everything = np.arange(len(cases))
    off = np.concatenate([[0], np.cumsum([c.col.nz for c in cases])])
    assert off[-1] >= 12 * cus and off[-1] % 2 == 1
    for mol in (1, 0):
        many = blocks(everything, mol)
        for i in (0, 1, len(cases) // 2, len(cases) - 1):
            few = blocks(everything[i:i + 1], mol)
            s = slice(off[i], off[i + 1])
            for a, b in zip(many[:6], few[:6]):
                assert np.array_equal(a[s], b)
        col = cases[-1].col
        J = O.jac_blocks(net, y0[-1], col.M, few[6])
        assert np.array_equal(few[0], J)
        for a, b in zip(few[1:4], O.lhs_blocks(col, y0[-1], dt[-1], J, bool(mol))):
            assert np.array_equal(a, b)
