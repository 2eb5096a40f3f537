"""Layers whose widths fill neither the narrow kernel's four-channel pieces nor
its 16-column tiles, against the fp64 oracle."""
import numpy as np
import pytest
import torch

from gpu_util import DEV, needs_gpu
from test_gpu_conv import _check_layer, _conv_raw, _module, _tiny
from trispconv_amd.pytorch.indices import generate_subm_indice_pairs

pytestmark = [pytest.mark.gpu, needs_gpu]


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("c_in,c_out,k", [(1, 1, 3), (2, 17, 3), (3, 32, 5), (5, 16, 3), (6, 3, 3),
                                          (7, 40, 1), (9, 15, 3), (13, 33, 3), (96, 20, 1),
                                          (64, 20, 3)])
def test_ragged_widths(c_in, c_out, k, dtype):
    """Every remainder of C_in mod 4, one to several column tiles, the identity
    map and 125 slots, and row counts from less than one piece of features
    (read element by element) over partial and whole 16-row waves and 64-row
    workgroups up to several.  The same features aligned to their elements
    only, through the C ABI, give the same bits; and with every other row
    infinite, the finite rows of a 1x1x1 layer must not see what an unaligned
    piece read past their own end."""
    shape = (12, 11, 13)
    for n in (1, 2, 5, 16, 63, 64, 65, 700):
        idx = _tiny(3, shape, 1, n)
        feats = np.random.default_rng(n).standard_normal((n, c_in)).astype(np.float32)
        m = _module("subm", c_in, c_out, k, dtype=dtype, seed=c_in + c_out)
        y = _check_layer(m, feats, idx, shape, 1, dtype, what=f"ragged {c_in}->{c_out} n={n}")
        data = generate_subm_indice_pairs(torch.from_numpy(idx).to(DEV), shape, 1, k)
        nbr = data.neighbour_map(n, DEV)
        room = torch.empty(n * c_in + 1, dtype=dtype, device=DEV)
        odd = room[1:].view(n, c_in)
        odd.copy_(torch.from_numpy(feats))
        z = _conv_raw(odd, m._packed_weight(dtype), m.bias, nbr, None, 0, n, 0)
        assert torch.equal(z, y.features), (n, c_in, c_out)
        if k == 1 and n > 1:
            odd[::2] = float("inf")
            z = _conv_raw(odd, m._packed_weight(dtype), m.bias, nbr, None, 0, n, 0)
            assert torch.equal(z[1::2], y.features[1::2])
            assert not torch.isfinite(z[::2]).any()


@pytest.mark.parametrize("c_in,c_out", [(12, 48), (5, 40), (7, 64), (20, 96)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
def test_column_tiles_per_wave(c_in, c_out, dtype):
    """Row counts around the lines between one, two, three and four column
    tiles per wave: the tiles of a wave share its gathers and nothing else, so
    a row's bits do not depend on how many there are (the first 2900 rows of
    each layer against a 2900-row layer, which has one, on the same map)."""
    shape = (40, 44, 48)
    for n in (12_736, 12_864, 25_536, 25_664, 38_336, 38_464):
        idx = _tiny(9, shape, 1, n)
        feats = np.random.default_rng(n).standard_normal((n, c_in)).astype(np.float32)
        m = _module("subm", c_in, c_out, 3, dtype=dtype, seed=c_in)
        y = _check_layer(m, feats, idx, shape, 1, dtype, rows=2000, what=f"tiles {c_out} n={n}")
        nbr = generate_subm_indice_pairs(torch.from_numpy(idx).to(DEV), shape, 1, 3).neighbour_map(n, DEV)
        few = nbr[:, :2900].contiguous()
        f = torch.from_numpy(feats).to(DEV).to(dtype)
        z = _conv_raw(f, m._packed_weight(dtype), m.bias, few, None, 0, 2900, 0)
        assert torch.equal(z, y.features[:2900])
