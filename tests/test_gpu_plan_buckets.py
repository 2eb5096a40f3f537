"""The execution order of built maps: sorted by slot mask, the map with it."""
import pytest
import torch

from gpu_util import DEV, needs_gpu
from test_gpu_conv import _tiny
from trispconv_amd.pytorch import indices as I
from trispconv_amd.pytorch.indices import generate_subm_indice_pairs

pytestmark = [pytest.mark.gpu, needs_gpu]


@pytest.mark.parametrize("k", [(2, 5, 1), (1, 3, 5), 3, (4, 7, 1), (1, 29, 1)])
@pytest.mark.parametrize("n,e", [(257, 16), (5120, 24), (5121, 24), (20_000, 128), (60_000, 48)])
def test_order_and_its_map(k, n, e, monkeypatch):
    """10 to 29 slots (two to four digit passes), up to nearly all rows sharing
    their masks' leading nine bits (of 20k sparse voxels 18k have the centre slot
    alone): the order is a permutation of the rows, the map and its masks are
    permuted by it, each tile is sorted by mask and columns with equal masks keep
    their order in it (the whole order: test_gpu_plan_order.py)."""
    monkeypatch.setattr(I, "_PLAN_MIN_BYTES", 0)
    monkeypatch.setattr(I, "_PLAN_MIN_ROWS", 0)
    idx = _tiny(n, (e, e, e), 1, n)
    data = generate_subm_indice_pairs(torch.from_numpy(idx).to(DEV), (e, e, e), 1, k)
    K = data.K
    order = data.execution_order(n, DEV, 256, eager=True).long()
    assert torch.equal(order.sort().values, torch.arange(n, device=DEV))
    nbr = data.neighbour_map(n, DEV)
    assert torch.equal(data.ordered_map(), nbr[:, order])
    bits = ((nbr >= 0).long() << torch.arange(K, device=DEV)[:, None]).sum(0)
    m = bits[order]
    row = data.ordered_map().as_strided((n,), (1,), data.ordered_map().storage_offset() + K * n)
    assert torch.equal(row.long() & 0xffffffff, m)
    rank = torch.empty(n, dtype=torch.long, device=DEV)
    rank[data._cols_row.long()] = torch.arange(n, device=DEV)  # column of each row
    cols = rank[order]
    for t in range(0, n, 256):
        mt, ct = m[t:t + 256], cols[t:t + 256]
        assert (mt.diff() >= 0).all()
        same = mt.diff() == 0
        assert (ct.diff()[same] > 0).all()
