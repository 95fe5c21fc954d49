"""Rate constants of a batch and of its columns alone, bit for bit, at the
numbers of layers where a workgroup starts to take two, four and eight of them
and where a layer's pairs are split over workgroups."""
import numpy as np
import pytest

from vulcan_amd import workloads as W
from vulcan_amd.config import Config

gpu = pytest.mark.gpu


@gpu
@pytest.mark.parametrize('per_cu', [1, 2, 5.5, 11, 22])
@pytest.mark.parametrize('extra', [-1, 1])
def test_rates_do_not_depend_on_the_batch(per_cu, extra):
    import torch
    if not torch.cuda.is_available():
        pytest.skip('no HIP device')
    from vulcan_amd.device import ColumnBatch, DevicePlan
    net = W.full_network()
    layers = int(per_cu * torch.cuda.get_device_properties(0).multi_processor_count) + extra
    nz = [50] * (layers // 50 - 1)
    nz.append(layers - sum(nz))
    plan, cases = DevicePlan(net), {n: W.small_case(nz=n, net=net) for n in set(nz)}

    def rates(some):
        b = ColumnBatch(plan, [cases[n].col for n in some], [cases[n].y0 for n in some], Config(), tune=False)
        k = b.k.cpu().numpy()
        b.close()
        return k

    k = rates(nz)
    assert k.shape[0] == layers
    assert np.array_equal(k[:50], rates(nz[:1])) and np.array_equal(k[-nz[-1]:], rates(nz[-1:]))
