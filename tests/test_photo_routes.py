"""Radiative transfer of batches whose size alone moves them to other kernels,
against their first two columns alone, bit for bit: the photolysis rates of many
layers with few and with many bins, and the fluxes of batches with so many bins
in all that a thread takes one each (short columns, columns whose LDS lets two
workgroups or one share a CU), beside the next smaller batch that does not."""
import numpy as np
import pytest

gpu = pytest.mark.gpu


def _update(torch, nz, nb, period):
    """Two updates of columns whose layers repeat every `period`; the rows of the
    first and of the last two columns."""
    from vulcan_amd import photo as P
    from vulcan_amd import workloads as W
    from vulcan_amd.device import DeviceColumns, DevicePlan
    net = W.small_network()
    rng = np.random.default_rng(nb)
    nabs, nbr = 5, 18
    tab = P.PhotoTables(bins=np.linspace(100., 300., nb), din12=max(1, nb // 3), sflux_top=10.0 ** rng.uniform(2, 5, nb),
                        abs_sp=[2, 7, 11, 20, 3], abs_T=[-1] * nabs, cross=10.0 ** rng.uniform(-21, -18, (nabs, nb)),
                        cross_T=np.zeros((0, 0, nb)), scat_sp=[1, 5], cross_scat=10.0 ** rng.uniform(-25, -22, (2, nb)),
                        br_col=[2 * q for q in range(nbr)], br_T=[-1] * nbr, cross_J=10.0 ** rng.uniform(-21, -18, (nbr, nb)),
                        cross_J_T=np.zeros((0, 0, nb)), dbin1=0.1, dbin2=2., cos_sl=0.669, edd=0.5, f_diurnal=1.,
                        flux_atol=1.)
    y = torch.as_tensor(10.0 ** rng.uniform(5, 13, (period, net.ni)), device='cuda')
    dz = torch.as_tensor(rng.uniform(1e5, 1e6, period), device='cuda')
    plan, cols = DevicePlan(net), DeviceColumns(nz)
    ph = P.DevicePhoto(plan, cols, tab)
    again = -(-cols.L // period)
    yd, dzd = y.repeat(again, 1)[:cols.L].contiguous(), dz.repeat(again)[:cols.L].contiguous()
    k = torch.zeros((cols.L, net.nr), dtype=torch.float64, device='cuda')
    for _ in range(2):
        ph.update(yd, yd / yd.sum(dim=1, keepdim=True), dzd, k, force=True)
    torch.cuda.synchronize()
    lay, lev = [(n, sum(nz[:2]) + n, sum(nz[-2:]) + n) for n in (0, 2)]
    out = []
    for what, rows in [(w, lev) for w in range(4)] + [(4, lay)]:
        a = ph.read(what)
        out += [a[:rows[1]], a[-rows[2]:]]
    out += [k[:lay[1], :2 * nbr].cpu().numpy(), k[-lay[2]:, :2 * nbr].cpu().numpy()]
    ph.close()
    assert (out[-1][:, ::2] > 0).all()
    return out


def _compare(nz, count, nb):
    import torch
    if not torch.cuda.is_available():
        pytest.skip('no HIP device')
    few, many = (_update(torch, nz * n, nb, sum(nz)) for n in (1, count))
    for a, b in zip(few, many):
        assert np.array_equal(a, b)


@gpu
@pytest.mark.parametrize('nz,count,nb', [([64, 41], 20, 511), ([64, 41], 20, 512), ([64, 41], 20, 3),
                                         ([64, 41], 20, 2600), ([64, 41], 11, 2601)])
def test_rates_of_many_layers(nz, count, nb):
    _compare(nz, count, nb)


@gpu
@pytest.mark.parametrize('nz,per_bin,nb', [([8, 5], 64000, 131), ([31, 2], 248000, 700), ([63, 40], 504000, 2588),
                                           ([213, 200], 180000, 700), ([320, 31], 90000, 1000), ([416, 3], 90000, 2588)])
@pytest.mark.parametrize('beyond', [0, 1])
def test_fluxes_of_many_bins(nz, per_bin, nb, beyond):
    _compare(nz, (per_bin - 1) // (2 * nb) + beyond, nb)


@gpu
def test_half_a_million_layers():
    """More groups of eight layers than a grid is long in y (65 535)."""
    _compare([128, 130], 2040, 5)


@gpu
@pytest.mark.parametrize('nz', [[3] * 9, [8] * 5, [17, 2, 3, 30, 5, 2]])
def test_columns_that_are_not_due(nz):
    """Each column due alone, beside columns that share its groups of eight
    layers: its own fluxes and rates as all columns' update leaves them, nothing
    written for the others."""
    import torch
    if not torch.cuda.is_available():
        pytest.skip('no HIP device')
    from vulcan_amd import _lib
    from vulcan_amd import photo as P
    from vulcan_amd import workloads as W
    from vulcan_amd.device import DeviceColumns, DevicePlan
    net, nb, nbr = W.small_network(), 300, 6
    rng = np.random.default_rng(len(nz))
    tab = P.PhotoTables(bins=np.linspace(100., 300., nb), din12=100, sflux_top=10.0 ** rng.uniform(2, 5, nb),
                        abs_sp=[2, 7, 11], abs_T=[-1] * 3, cross=10.0 ** rng.uniform(-21, -18, (3, nb)),
                        cross_T=np.zeros((0, 0, nb)), scat_sp=[1], cross_scat=10.0 ** rng.uniform(-25, -22, (1, nb)),
                        br_col=[2 * q for q in range(nbr)], br_T=[-1] * nbr, cross_J=10.0 ** rng.uniform(-21, -18, (nbr, nb)),
                        cross_J_T=np.zeros((0, 0, nb)), dbin1=0.1, dbin2=2., cos_sl=0.669, edd=0.5, f_diurnal=1.,
                        flux_atol=1.)
    plan, cols = DevicePlan(net), DeviceColumns(nz)
    y = torch.as_tensor(10.0 ** rng.uniform(5, 13, (cols.L, net.ni)), device='cuda')
    dz = torch.as_tensor(rng.uniform(1e5, 1e6, cols.L), device='cuda')
    ymix = y / y.sum(dim=1, keepdim=True)
    arrays = [(w, 1 if w < 4 else 0) for w in range(5)]

    def rows(c, more):   # one level more than layers, column by column
        o = sum(nz[:c]) + more * c
        return slice(o, o + nz[c] + more)

    def run(due):
        ph = P.DevicePhoto(plan, cols, tab)
        k = torch.zeros((cols.L, net.nr), dtype=torch.float64, device='cuda')
        if due is None:
            ph.update(y, ymix, dz, k, force=True)
        else:
            st = np.zeros(len(nz), _lib.COLSTATE_DTYPE)
            st['longdy'], st['done'] = 1., np.arange(len(nz)) != due
            ph.update(y, ymix, dz, k, state=torch.as_tensor(st.view(np.uint8).reshape(-1), device='cuda'), force=False)
        torch.cuda.synchronize()
        out = [ph.read(w) for w, _ in arrays] + [k.cpu().numpy()]
        ph.close()
        return out

    every = run(None)
    for due in range(len(nz)):
        for a, b, (_, more) in zip(run(due), every, arrays + [(5, 0)]):
            for c in range(len(nz)):
                want = b[rows(c, more)] if c == due else 0.0
                assert np.array_equal(a[rows(c, more)], np.broadcast_to(want, b[rows(c, more)].shape)), (due, c)
