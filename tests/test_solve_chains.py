"""The chain solves around every edge of their layout: the 16-species tiles,
one, two or three columns per lane, waves whose last rows or all rows lie past
the block, chains shorter than, as long as and longer than the loads in flight
(1, 2 and 4 layers), without and with a refinement (which adds into the
solution), against a dense solve in float64.

Tolerance: as for the factorisation, condition numbers of at most a few
hundred and n <= 160 give n eps cond < 1e-11 of the solution's largest entry."""
import numpy as np
import pytest

from vulcan_amd import _lib
from test_factor_pivots import TOL, _dense, _network, _system

gpu = pytest.mark.gpu


@gpu
@pytest.mark.parametrize('refine', [0, 1])
@pytest.mark.parametrize('ni', [1, 2, 15, 16, 17, 31, 32, 33, 48, 49, 63, 64, 65, 81, 93, 96, 97, 112,
                                113, 127, 128, 129, 144, 145, 150, 160])
def test_chain_solves(ni, refine):
    import torch
    if not torch.cuda.is_available():
        pytest.skip('no HIP device')
    from vulcan_amd.device import DeviceColumns, DevicePlan, dptr, stream_handle
    nz = [2, 3, 4, 5, 6, 7, 8, 15, 16, 17, 18, 19, 33]
    D, Ls, Us, b, off = _system(ni, nz, 'diagonal', 11 * ni)
    # couplings across the ends of a column are never used
    Ls[off[:-1]] = Us[off[1:] - 1] = np.nan
    ref = np.concatenate([_dense(D[o:p], Ls[o:p], Us[o:p], b[o:p]) for o, p in zip(off[:-1], off[1:])])
    lib = _lib.load()
    plan, cols = DevicePlan(_network(ni)), DeviceColumns(nz)
    d = [torch.as_tensor(a, device='cuda') for a in (D, Ls, Us, b)]
    x = torch.empty_like(d[3])
    info = torch.full((len(nz),), -1, dtype=torch.int32, device='cuda')
    _lib.check(lib.vk_plan_set_factor_variant(plan.handle, 1), 'vk_plan_set_factor_variant')
    _lib.check(lib.vk_block_solve_system(plan.handle, cols.handle, *[dptr(t) for t in d], dptr(x), refine, dptr(info),
                                         stream_handle()), 'vk_block_solve_system')
    assert not info.cpu().numpy().any()
    assert np.abs(x.cpu().numpy() - ref).max() < TOL * np.abs(ref).max()


@gpu
@pytest.mark.parametrize('ni', [1, 7, 63, 64, 65, 95, 96, 97, 127, 128, 129, 153, 160])
@pytest.mark.parametrize('nz', [[2], [9], [2, 3, 17, 8, 5]])
def test_cyclic_reduction_solves(ni, nz):
    """The row-group sweeps at the edges of their chunk sizes (8, 12, 16 and
    20 entries of a row per thread) and of the groups of 32 rows, with one
    column (its last level in one launch up to 96 species) and several."""
    import torch
    if not torch.cuda.is_available():
        pytest.skip('no HIP device')
    from vulcan_amd.device import DeviceColumns, DevicePlan, dptr, stream_handle
    D, Ls, Us, b, off = _system(ni, nz, 'diagonal', 13 * ni + len(nz))
    ref = np.concatenate([_dense(D[o:p], Ls[o:p], Us[o:p], b[o:p]) for o, p in zip(off[:-1], off[1:])])
    lib = _lib.load()
    plan, cols = DevicePlan(_network(ni)), DeviceColumns(nz)
    d = [torch.as_tensor(a, device='cuda') for a in (D, Ls, Us, b)]
    x = torch.empty_like(d[3])
    info = torch.full((len(nz),), -1, dtype=torch.int32, device='cuda')
    _lib.check(lib.vk_plan_set_factor_variant(plan.handle, 4), 'vk_plan_set_factor_variant')
    for refine in (0, 1):
        x.zero_()
        _lib.check(lib.vk_block_solve_system(plan.handle, cols.handle, *[dptr(t) for t in d], dptr(x), refine,
                                             dptr(info), stream_handle()), 'vk_block_solve_system')
        assert not info.cpu().numpy().any()
        assert np.abs(x.cpu().numpy() - ref).max() < TOL * np.abs(ref).max()
