"""A strided build's IndiceData pickles and copies, and what it leads to is
the same afterwards."""
import copy
import pickle

import pytest
import torch

from gpu_util import DEV, needs_gpu
from test_gpu_conv import _tiny
from trispconv_amd.pytorch import indices as I
from trispconv_amd.pytorch.indices import (generate_inverse_indice_pairs,
                                           generate_strided_indice_pairs, inverse_pairs_for)

pytestmark = [pytest.mark.gpu, needs_gpu]


@pytest.mark.parametrize("way", [lambda d: pickle.loads(pickle.dumps(d)), copy.deepcopy],
                         ids=["pickle", "deepcopy"])
@pytest.mark.parametrize("read", [False, True])
def test_round_trip(way, read, monkeypatch):
    idx = torch.from_numpy(_tiny(5, (14, 15, 16), 1, 700)).to(DEV)
    made = [generate_strided_indice_pairs(idx, (14, 15, 16), 1, 3, 2, 1) for _ in range(2)]
    if read:  # pair_num and the lists made before
        made[0].pairs_in  # noqa: B018
    got, want = way(made[0]), made[1]
    assert torch.equal(got.pair_num, want.pair_num)
    assert torch.equal(got.out_indices, want.out_indices)
    for a, b in zip(got.pairs_in + got.pairs_out, want.pairs_in + want.pairs_out):
        assert torch.equal(a, b)
    assert not inverse_pairs_for(got, 64, 64, torch.float16)._grouped
    monkeypatch.setattr(I, "_GROUP_MIN_WORK", 0)
    up = inverse_pairs_for(got, 64, 64, torch.float16)
    assert up._grouped
    plain = generate_inverse_indice_pairs(want)
    assert torch.equal(up.out_indices, plain.out_indices)
    assert torch.equal(up.neighbour_map(len(up.out_indices), DEV), plain.neighbour_map(len(up.out_indices), DEV))
    again = way(up)
    assert all(torch.equal(a, b) for a, b in zip(again.pairs_out, plain.pairs_out))
