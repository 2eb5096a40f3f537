"""The int64 pair lists made from the padded tables in one launch per 64 slots."""
import ctypes

import pytest
import torch

import trispconv_amd._lib as L
from gpu_util import DEV, needs_gpu

pytestmark = [pytest.mark.gpu, needs_gpu]


@pytest.mark.parametrize("K,cap", [(1, 1), (27, 1023), (27, 1025), (64, 700), (65, 2049), (125, 300)])
def test_lists_are_the_table_slices(K, cap):
    """Empty, full and partial slots; one slot, 64 (one launch) and more; sizes
    on both sides of a block's 1024 entries; nothing written past the lists."""
    g = torch.Generator().manual_seed(K * cap)
    tables = torch.randint(-1, 1 << 30, (2, K, cap), generator=g, dtype=torch.int32).to(DEV)
    sizes = [int(v) for v in torch.randint(0, cap + 1, (K,), generator=g)]
    sizes[0], sizes[-1] = cap, cap
    if K > 2:
        sizes[1] = 0
    total = sum(sizes)
    out = torch.full((2, total + 8), -7, dtype=torch.int64, device=DEV)
    L.check(L.lib().tsc_pair_lists(tables[0].data_ptr(), tables[1].data_ptr(), K, cap,
                                   (ctypes.c_int64 * K)(*sizes), out[0].data_ptr(),
                                   out[1].data_ptr(), L.stream_of(tables)), "lists")
    for i in range(2):
        want = torch.cat([tables[i, k, :c].long() for k, c in enumerate(sizes)])
        assert torch.equal(out[i, :total], want)
        assert (out[i, total:] == -7).all()
    sizes[0] = cap + 1
    with pytest.raises(ValueError):
        L.check(L.lib().tsc_pair_lists(tables[0].data_ptr(), tables[1].data_ptr(), K, cap,
                                       (ctypes.c_int64 * K)(*sizes), out[0].data_ptr(),
                                       out[1].data_ptr(), L.stream_of(tables)), "lists")
