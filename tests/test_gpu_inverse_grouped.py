"""Inverse maps with their columns grouped by the slots they can use."""
import numpy as np
import pytest
import torch

import trispconv.pytorch as spconv
from gpu_util import DEV, needs_gpu, say
from test_gpu_pairs import _inverse, _strided, _tiny
from trispconv_amd import _lib as L
from trispconv_amd.pytorch import indices as I

pytestmark = [pytest.mark.gpu, needs_gpu]


@pytest.mark.parametrize("k,s,p,d", [(3, 2, 1, 1), (2, 2, 0, 1), ((3, 1, 1), (2, 1, 1), 0, 1),
                                     (3, 3, 1, 1), (3, (1, 2, 4), (0, 1, 1), (1, 2, 1)), (3, 4, 1, 1)])
@pytest.mark.parametrize("n", [1, 255, 1023, 1025, 4200])
def test_grouped_columns_hold_the_row_order_map(k, s, p, d, n, monkeypatch):
    """Against the oracle (pair lists, coordinates) and, for the map itself,
    against the inverse in row order: the columns' rows are a permutation, the
    map read through them is the row-order map, and the columns' slot sets
    come in one run per residue class (2 to 64 of them), longest sets first
    (rows at the grid's border may lack some of their class's slots).  Row
    counts below, at and past a count block's 1024."""
    shape, B = (17, 18, 21), 2
    idx = _tiny(n, shape, B, n)
    g, e = _strided(idx, shape, B, k, s, p, d, "forward")
    plain = _inverse(g, e, "row order")
    n_out = len(plain.out_indices)
    monkeypatch.setattr(I, "_GROUP_MIN_WORK", 0)
    got = _inverse(g, e, "grouped")
    assert got._grouped and not plain._grouped
    if n_out == 0:
        return
    rows = got._cols_row.cpu().numpy()
    assert np.array_equal(np.sort(rows), np.arange(n_out))
    assert torch.equal(got.neighbour_map(n_out, DEV), plain.neighbour_map(n_out, DEV))
    st, pd = g.stride, g.padding
    c = plain.out_indices.cpu().numpy()[rows][:, 1:]
    cls = np.ravel_multi_index(tuple(((c + pd) % st).T), st)
    runs = cls[np.concatenate([[True], cls[1:] != cls[:-1]])]
    assert len(runs) == len(np.unique(runs))  # each class in one run
    assert all((np.diff(rows[cls == v]) > 0).all() for v in runs)  # rows ascend within it
    # the slots of a class: per axis, the kernel offsets that land on its residue
    ks, dil = np.array(g.kernel_size), np.array(g.dilation)
    hits = [[sum(o * dil[a] % st[a] == r for o in range(ks[a])) for r in range(st[a])] for a in range(3)]
    slots = [np.prod([hits[a][r] for a, r in enumerate(np.unravel_index(v, st))]) for v in runs]
    say("classes", len(runs), slots)
    assert (np.diff(slots) <= 0).all()
    most = np.array([int((got._map_cols >= 0).sum(0).cpu().numpy()[cls == v].max()) for v in runs])
    assert (most <= slots).all()


@pytest.mark.parametrize("n", [300, 9000, 60000])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_inverse_layer_is_the_same_bits_grouped_or_not(n, dtype, monkeypatch):
    """Through the modules: layers of the slot-split, direct-to-LDS, register
    gather and narrow kernels, on the first use, the second (which adds the
    columns' masks where the rows are many enough) and the third."""
    monkeypatch.setattr(I, "_PLAN_MIN_BYTES", 1 << 20)
    shape = (40, 40, 40)
    idx = torch.from_numpy(_tiny(3, shape, 1, n)).to(DEV)
    for c_mid, c_out in ((64, 32), (128, 64), (48, 32), (32, 16), (48, 20)):
        torch.manual_seed(c_mid)
        down = spconv.SparseConv3d(32, c_mid, 3, stride=2, padding=1, indice_key="k").to(DEV).to(dtype)
        up = spconv.SparseInverseConv3d(c_mid, c_out, 3, indice_key="k").to(DEV).to(dtype)
        f = torch.randn(n, 32, device=DEV).to(dtype)
        outs = []
        for line in (1 << 60, 1):
            monkeypatch.setattr(I, "_GROUP_MIN_WORK", line)
            y = down(spconv.SparseConvTensor(f, idx, list(shape), 1))
            z = up(y)
            for use in range(2):
                assert torch.equal(z.features, up(y).features)
            inv = y.indice_dict["k"]._inverse_cache
            assert inv._grouped == (line == 1 and c_out % 32 == 0)
            if inv._grouped and n == 60000:
                assert inv._map_masks
            outs.append(z)
        assert torch.equal(outs[0].indices, outs[1].indices)
        assert torch.equal(outs[0].features, outs[1].features)
