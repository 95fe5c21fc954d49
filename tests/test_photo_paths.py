"""The radiative transfer's kernels for short and long columns, few and many
layers, against each other: the same columns give the same bits whichever
path the batch takes (columns beyond 416 layers run a thread per bin; the
photolysis rates take one, two or four layers per workgroup by the number of
layers, and the actinic flux from memory beyond 10 400 bins)."""
import numpy as np
import pytest

gpu = pytest.mark.gpu


def _tables(nb, L, rng_seed, nabs=37, nbr=11, nT=3):
    """Random spectra; per-layer tables of the first layers do not depend on L."""
    from vulcan_amd import photo as P
    rng = np.random.default_rng(rng_seed)
    cross = 10.0 ** rng.uniform(-22, -16, (nabs, nb))
    cross_J = 10.0 ** rng.uniform(-22, -16, (nbr, nb))
    sc = 10.0 ** rng.uniform(-26, -20, (2, nb))
    sfl = 10.0 ** rng.uniform(0, 5, nb)
    f = np.random.default_rng(99).uniform(0.5, 1.5, (8000, 1))[:L]
    abs_T = [-1] * nabs
    abs_T[5], abs_T[0], abs_T[36] = 0, 1, 2
    br_T = [-1] * nbr
    br_T[2], br_T[10] = 0, 1
    return P.PhotoTables(bins=np.linspace(10., 600., nb), din12=max(1, nb // 2), sflux_top=sfl,
                         abs_sp=[int(i) for i in rng.integers(0, 28, nabs)], abs_T=abs_T, cross=cross,
                         cross_T=np.stack([cross[a] * f for a in (5, 0, 36)]), scat_sp=[1, 3], cross_scat=sc,
                         br_col=[2 * q for q in range(nbr)], br_T=br_T, cross_J=cross_J,
                         cross_J_T=np.stack([cross_J[b] * f for b in (2, 10)]), dbin1=0.1, dbin2=2., cos_sl=0.669,
                         edd=0.5, f_diurnal=1., flux_atol=1.)


def _run(torch, nz, nb):
    from vulcan_amd import _lib
    from vulcan_amd import photo as P
    from vulcan_amd import workloads as W
    from vulcan_amd.device import DeviceColumns, DevicePlan
    net = W.small_network()
    plan, cols = DevicePlan(net), DeviceColumns(nz)
    L = cols.L
    ph = P.DevicePhoto(plan, cols, _tables(nb, L, 3))
    rng = np.random.default_rng(5)
    y = 10.0 ** rng.uniform(5, 16, (8000, net.ni))[:L]
    up = lambda a: torch.as_tensor(np.ascontiguousarray(a), device='cuda')
    dz = up(rng.uniform(1e5, 1e7, 8000)[:L])
    yd, md = up(y), up(y / y.sum(axis=1, keepdims=True))
    k = torch.zeros((L, net.nr), dtype=torch.float64, device='cuda')
    st = torch.zeros((len(nz), _lib.COLSTATE_DTYPE.itemsize), dtype=torch.uint8, device='cuda')
    for _ in range(2):                       # the second update starts from the first one's upward flux
        ph.update(yd, md, dz, k, state=st, force=True)
    torch.cuda.synchronize()
    out = {what: ph.read(what) for what in range(5)}
    out['k'] = k.cpu().numpy()
    out['change'] = st.cpu().numpy().reshape(-1).view(_lib.COLSTATE_DTYPE)['aflux_change'].copy()
    ph.close()
    return out


@gpu
@pytest.mark.parametrize('nb,nz,more', [
    (131, [33, 160, 2, 97, 224], [417]),           # long columns: a thread per bin
    (7, [32, 33, 64, 65], [416]), (257, [96, 97], [161]),
    (300, [40, 3], [64] * 16 + [7]),               # two layers per workgroup
    (300, [40, 3], [64] * 33 + [7])])              # four
def test_paths_agree_bitwise(nb, nz, more):
    import torch
    if not torch.cuda.is_available():
        pytest.skip('no HIP device')
    a, b = _run(torch, nz, nb), _run(torch, nz + more, nb)
    L, lev = sum(nz), sum(nz) + len(nz)
    for what in range(4):
        assert np.array_equal(a[what], b[what][:lev]), what
    assert np.array_equal(a[4], b[4][:L])
    assert np.array_equal(a['k'], b['k'][:L])
    assert np.array_equal(a['change'], b['change'][:len(nz)])
    rates = a['k'][:, ::2][:, :11]                 # optically thick layers may underflow to zero
    assert np.isfinite(rates).all() and (rates >= 0).all() and (rates[nz[0] - 1] > 0).all()


@gpu
def test_spectra_beyond_lds_in_the_loop():
    """10 403 bins: vk_photo_update refuses them, the integration's own
    refresh reads the actinic flux from memory; one column alone against the
    same column beside a longer one."""
    import torch
    if not torch.cuda.is_available():
        pytest.skip('no HIP device')
    from vulcan_amd import _lib
    from vulcan_amd import photo as P
    from vulcan_amd import workloads as W
    from vulcan_amd.device import ColumnBatch, DevicePlan
    nb, got = 10403, []
    for nzs in ([7], [7, 417]):
        cs = [W.small_case(nz) for nz in nzs]
        b = ColumnBatch(DevicePlan(cs[0].net), [c.col for c in cs], [c.y0 for c in cs], cs[0].cfg, tune=False)
        ph = P.DevicePhoto(b.plan, b.layout, _tables(nb, b.layout.L, 4, nabs=37))
        with pytest.raises(_lib.VulcanAmdError):
            ph.update(b.y, b.ymix, b.dz, b.k, state=b.state, force=True)
        b.attach_photo(ph, 1, 1)
        b.integrate(1, use_conv=False)
        torch.cuda.synchronize()
        got.append(b.k.cpu().numpy()[:7].copy())
        b.attach_photo(None, 1, 1)
        ph.close()
        b.close()
    assert np.array_equal(got[0], got[1])
    assert np.isfinite(got[0]).all() and (got[0][6, ::2][:11] > 0).all()
