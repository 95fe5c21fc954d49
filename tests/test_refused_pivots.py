"""Blocks that refuse the diagonal as pivots and blocks that only just do not.

Which inversion ran is seen from its bits.  With the diagonal as pivots,
scaling a block's rows and columns by powers of two scales every intermediate
exactly, so the inverse is that of the unscaled block to the last bit; searched
pivots move with the scales of the rows, and the rounding with them.

Refused blocks may cost the attempt, but not a second pass of the whole launch:
a batch with one refusing chain is no slower than one in which every chain
refuses (times of one process beside each other; a second pass is 1.4 to 1.5
times as long)."""
import numpy as np
import pytest

from vulcan_amd import _lib
from test_factor_pivots import _network

gpu = pytest.mark.gpu


def _setup(ni, nz):
    import torch
    if not torch.cuda.is_available():
        pytest.skip('no HIP device')
    from vulcan_amd.device import DeviceColumns, DevicePlan
    return torch, _lib.load(), DevicePlan(_network(ni)), DeviceColumns(nz)


def _inverses(ctx, variant, D):
    """The inverse of every block of D, all couplings zero: from the chain
    factorisation, or column by column from cyclic reduction's solves."""
    torch, lib, plan, cols = ctx
    from vulcan_amd.device import dptr, stream_handle
    L, ni, _ = D.shape
    _lib.check(lib.vk_plan_set_factor_variant(plan.handle, variant), 'vk_plan_set_factor_variant')
    d = torch.as_tensor(np.ascontiguousarray(D), device='cuda')
    zero = torch.zeros((L, ni), dtype=torch.float64, device='cuda')
    if variant != 4:
        X = torch.empty_like(d)
        _lib.check(lib.vk_block_factor(plan.handle, cols.handle, dptr(d), dptr(zero), dptr(zero), dptr(X), None,
                                       stream_handle()), 'vk_block_factor')
        return X.cpu().numpy().transpose(0, 2, 1)
    out = np.empty_like(D)
    b, x = torch.empty_like(zero), torch.empty_like(zero)
    for j in range(ni):
        b.zero_()
        b[:, j] = 1.0
        _lib.check(lib.vk_block_solve_system(plan.handle, cols.handle, dptr(d), dptr(zero), dptr(zero), dptr(b), dptr(x),
                                             0, None, stream_handle()), 'vk_block_solve_system')
        out[:, :, j] = x.cpu().numpy()
    return out


def _exact_inverse(A):
    """Gauss-Jordan with partial pivoting in extended precision."""
    n = len(A)
    W = np.concatenate([A.astype(np.longdouble), np.eye(n, dtype=np.longdouble)], axis=1)
    for k in range(n):
        p = k + np.abs(W[k:, k]).argmax()
        W[[k, p]] = W[[p, k]]
        W[k] /= W[k, k]
        f = W[:, k].copy()
        f[k] = 0
        W -= f[:, None] * W[k]
    return W[:, n:]


def _blocks(ni, L, near, rng):
    """M-matrices (1 + near) I - P with P's rows summing to 1: the last pivots are
    small parts of their diagonal entries (1e-2 to 3e-8 for near 1e-4 to 1e-8)."""
    P = rng.random((L, ni, ni)) ** 4 + 1e-6
    P[:, range(ni), range(ni)] = 0.0
    P /= P.sum(axis=2, keepdims=True)
    return (1.0 + near) * np.eye(ni) - P


@gpu
@pytest.mark.parametrize('near', [1e-4, 1e-8])
@pytest.mark.parametrize('ni,nz', [(4, [3, 2]), (17, [5]), (33, [2, 4]), (48, [150]), (97, [3]), (112, [150]), (144, [3])])
@pytest.mark.parametrize('variant', [1, 2, 4])
def test_scaled_and_nearly_singular_blocks_keep_the_diagonal(variant, ni, nz, near):
    """Pivots down to 3e-8 of their entries are taken, and the inverse is as near
    the exact one as a stable elimination's: within 4 n eps cond."""
    if variant == 4 and ni > 48:
        nz = nz[:1]
    ctx = _setup(ni, nz)
    rng = np.random.default_rng(ni)
    D = _blocks(ni, sum(nz), near, rng)
    L = len(D)
    r, c = 2.0 ** rng.integers(-20, 21, (2, L, ni))
    X, Xs = _inverses(ctx, variant, D), _inverses(ctx, variant, D * r[:, :, None] * c[:, None, :])
    assert np.array_equal(Xs, X / r[:, None, :] / c[:, :, None])
    for l in {0, L // 2, L - 1}:
        ref = _exact_inverse(D[l])
        cond = np.abs(D[l]).sum(axis=1).max() * np.abs(ref).sum(axis=1).max()
        assert np.abs(X[l] - ref).max() <= 4 * ni * 2.2e-16 * cond * np.abs(ref).max()


@gpu
@pytest.mark.parametrize('ni,nz', [(17, [5]), (48, [150]), (97, [3])])
@pytest.mark.parametrize('variant', [1, 2, 4])
def test_refused_blocks_are_searched(variant, ni, nz):
    ctx = _setup(ni, nz)
    rng = np.random.default_rng(ni)
    D = np.roll(_blocks(ni, sum(nz), 1e-2, rng), 1, axis=1)
    r = 2.0 ** rng.integers(-20, 21, (len(D), ni))
    X, Xs = _inverses(ctx, variant, D), _inverses(ctx, variant, D * r[:, :, None])
    for l in range(len(D)):
        assert not np.array_equal(Xs[l], X[l] / r[l])
        assert np.allclose(X[l] @ D[l], np.eye(ni), atol=1e-9)


@gpu
@pytest.mark.parametrize('ni', [30, 93, 150])
@pytest.mark.parametrize('variant', [1, 2])
def test_one_refusing_chain_costs_no_second_pass(variant, ni):
    nz = [40] * 6
    torch, lib, plan, cols = _setup(ni, nz)
    from vulcan_amd.device import dptr, stream_handle
    rng = np.random.default_rng(ni)
    kept = _blocks(ni, sum(nz), 1.0, rng)
    every = np.roll(kept, 1, axis=1)
    one = kept.copy()
    one[0] = every[0]
    _lib.check(lib.vk_plan_set_factor_variant(plan.handle, variant), 'vk_plan_set_factor_variant')
    zero = torch.zeros((sum(nz), ni), dtype=torch.float64, device='cuda')
    D = [torch.as_tensor(a, device='cuda') for a in (every, one)]
    X = torch.empty_like(D[0])
    best = [np.inf, np.inf]
    for _ in range(10):
        for q in (0, 1):
            a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            a.record()
            _lib.check(lib.vk_block_factor(plan.handle, cols.handle, dptr(D[q]), dptr(zero), dptr(zero), dptr(X), None,
                                           stream_handle()), 'vk_block_factor')
            b.record()
            torch.cuda.synchronize()
            best[q] = min(best[q], a.elapsed_time(b))
    print('every chain refuses %.3f ms, one %.3f ms' % tuple(best), flush=True)
    assert best[1] < 1.15 * best[0]


@gpu
@pytest.mark.parametrize('every', [0, 2, 7, 9, 40])
@pytest.mark.parametrize('ni', [17, 97])
def test_cyclic_reduction_with_some_refusing(ni, every):
    """Refusals among the blocks that level 0 eliminates, none, fewer than one in
    eight or more (the later levels then search at once), and among the others
    too; columns of even and odd length, more blocks a launch than CUs."""
    from test_factor_pivots import TOL, _dense, _system
    nz = [40, 41, 2, 3] + [9] * 56
    torch, lib, plan, cols = _setup(ni, nz)
    from vulcan_amd.device import dptr, stream_handle
    D, Ls, Us, b, off = _system(ni, nz, 'diagonal', ni + every)
    for o, n in zip(off[:-1], nz):
        gone = np.arange(0 if n % 2 else 1, n, 2)
        for l in [*gone[::every]] if every else []:
            D[o + l] = np.roll(D[o + l], 1 + l % (ni - 1), axis=0)
        if every != 2 and n > 4:
            D[o + 6 - n % 2] = np.roll(D[o + 6 - n % 2], 1, axis=0)
    ref = np.concatenate([_dense(D[o:p], Ls[o:p], Us[o:p], b[o:p]) for o, p in zip(off[:-1], off[1:])])
    d = [torch.as_tensor(a, device='cuda') for a in (D, Ls, Us, b)]
    x = torch.empty_like(d[3])
    info = torch.full((len(nz),), -1, dtype=torch.int32, device='cuda')
    _lib.check(lib.vk_plan_set_factor_variant(plan.handle, 4), 'vk_plan_set_factor_variant')
    for _ in range(2):                       # the second time over the first one's inverses and marks
        x.zero_()
        _lib.check(lib.vk_block_solve_system(plan.handle, cols.handle, *[dptr(t) for t in d], dptr(x), 0, dptr(info),
                                             stream_handle()), 'vk_block_solve_system')
        assert not info.cpu().numpy().any()
        assert np.abs(x.cpu().numpy() - ref).max() < TOL * np.abs(ref).max()


@gpu
@pytest.mark.parametrize('ni', [112, 128])
def test_cyclic_reduction_attempts_refused_blocks_once(ni):
    """Blocks that refuse at their last pivots cost one level's attempt more than
    blocks that refuse at their first (an attempt a level is a third more)."""
    nz = [100]
    torch, lib, plan, cols = _setup(ni, nz)
    from vulcan_amd.device import dptr, stream_handle
    rng = np.random.default_rng(ni)
    kept = _blocks(ni, sum(nz), 1.0, rng)
    late = kept.copy()
    late[:, [ni - 2, ni - 1]] = late[:, [ni - 1, ni - 2]]
    _lib.check(lib.vk_plan_set_factor_variant(plan.handle, 4), 'vk_plan_set_factor_variant')
    zero = torch.zeros((sum(nz), ni), dtype=torch.float64, device='cuda')
    D = [torch.as_tensor(np.ascontiguousarray(a), device='cuda') for a in (np.roll(kept, 1, axis=1), late)]
    b, x = torch.ones_like(zero), torch.empty_like(zero)
    best = [np.inf, np.inf]
    for _ in range(8):
        for q in (0, 1):
            start, stop = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            for n in range(6):                # the first ones warm up the allocation
                if n == 1:
                    start.record()
                _lib.check(lib.vk_block_solve_system(plan.handle, cols.handle, dptr(D[q]), dptr(zero), dptr(zero), dptr(b),
                                                     dptr(x), 0, None, stream_handle()), 'vk_block_solve_system')
            stop.record()
            torch.cuda.synchronize()
            best[q] = min(best[q], start.elapsed_time(stop) / 5)
    print('refused at the first pivots %.3f ms, at the last %.3f ms' % tuple(best), flush=True)
    assert best[1] < 1.17 * best[0]
