"""Every pair list is a tensor of its own."""
import ctypes
import io

import pytest
import torch

import trispconv_amd._lib as L
from gpu_util import DEV, needs_gpu
from test_gpu_conv import _tiny
from trispconv_amd.pytorch.indices import (generate_inverse_indice_pairs,
                                           generate_strided_indice_pairs,
                                           generate_subm_indice_pairs)

pytestmark = [pytest.mark.gpu, needs_gpu]


def _builds(k=3, n=700):
    idx = torch.from_numpy(_tiny(5, (14, 15, 16), 1, n)).to(DEV)
    down = generate_strided_indice_pairs(idx, (14, 15, 16), 1, k, 2, 1)
    return [generate_subm_indice_pairs(idx, (14, 15, 16), 1, k), down, generate_inverse_indice_pairs(down)]


@pytest.mark.parametrize("k", [3, 5])
def test_storage_versions_and_size(k):
    """No two lists share memory or a version counter: holding or saving one
    holds that one, a write to one leaves what autograd saved of the others."""
    for data in _builds(k):
        lists = data.pairs_in + data.pairs_out
        full = [p for p in lists if p.numel()]
        assert len({p.untyped_storage().data_ptr() for p in full}) == len(full)
        for p in lists:
            assert p.untyped_storage().nbytes() == 8 * p.numel() and not p._is_view()
        kept = [p.clone() for p in lists]
        versions = [p._version for p in lists]
        big = max(range(len(lists)), key=lambda i: lists[i].numel())
        lists[big].add_(1)
        assert [p._version for i, p in enumerate(lists) if i != big] == \
            [v for i, v in enumerate(versions) if i != big]
        lists[big].resize_(lists[big].numel() + 64).fill_(-9)
        assert all(torch.equal(p, q) for i, (p, q) in enumerate(zip(lists, kept)) if i != big)
        f = io.BytesIO()
        one = min((p for p in full), key=lambda p: p.numel())
        torch.save(one, f)
        assert f.tell() < 8 * one.numel() + 4096


def test_gradients_through_one_list_after_a_write_to_another():
    data = _builds()[0]
    a, b = data.pairs_in[13], data.pairs_in[0]
    x = torch.randn(700, 4, device=DEV, requires_grad=True)
    y = x.index_select(0, a).mul(2).sum()
    b.zero_()
    y.backward()
    assert (x.grad == 2).all()


def test_an_assigned_list_stays_and_the_other_is_made():
    data = _builds()[1]
    want = [p.clone() for p in _builds()[1].pairs_out]
    mine = [torch.zeros(3, dtype=torch.long, device=DEV) for _ in range(27)]
    data.pairs_in = mine
    assert data.pairs_in is mine
    assert all(torch.equal(p, q) for p, q in zip(data.pairs_out, want))


@pytest.mark.parametrize("counts", ["short", "past", "negative"])
def test_counts_that_the_user_set(counts):
    """As slices of a slot's table: fewer slots, more entries than the table
    has, negative ends."""
    data = _builds()[1]
    cap = data._pin.shape[1]
    num = {"short": data.pair_num[:5], "past": torch.full((27,), cap + 9),
           "negative": torch.full((27,), -3)}[counts]
    want = [data._pin[k, :int(c)].long() for k, c in enumerate(num.tolist())]
    data.pair_num = num
    got = data.pairs_in
    assert len(got) == len(num) == len(data.pairs_out)
    assert all(torch.equal(p, q) for p, q in zip(got, want))


def test_counts_of_more_slots_than_there_are():
    data = _builds()[1]
    data.pair_num = torch.ones(28, dtype=torch.long)
    with pytest.raises(IndexError):
        data.pairs_in  # noqa: B018


@pytest.mark.parametrize("K,cap", [(1, 1), (27, 1025), (64, 700), (65, 2049)])
@pytest.mark.parametrize("sides", [(True, True), (True, False), (False, True)])
def test_entry(K, cap, sides):
    """Sides and slots without a destination are left out; nothing is written
    past a list."""
    g = torch.Generator().manual_seed(K * cap)
    tables = torch.randint(-1, 1 << 30, (2, K, cap), generator=g, dtype=torch.int32).to(DEV)
    sizes = [int(v) for v in torch.randint(0, cap + 1, (K,), generator=g)]
    sizes[0] = cap
    if K > 2:
        sizes[1] = 0
    out = [[torch.full((c + 4,), -7, dtype=torch.int64, device=DEV) for c in sizes] for _ in range(2)]
    ptr = [(ctypes.c_void_p * K)(*[t.data_ptr() if c else None for t, c in zip(side, sizes)]) for side in out]
    L.check(L.lib().tsc_pair_lists_each(tables[0].data_ptr(), tables[1].data_ptr(), K, cap,
                                        (ctypes.c_int64 * K)(*sizes), ptr[0] if sides[0] else None,
                                        ptr[1] if sides[1] else None, L.stream_of(tables)), "lists")
    for i in range(2):
        for k, c in enumerate(sizes):
            want = tables[i, k, :c].long() if sides[i] else torch.full((c,), -7, device=DEV)
            assert torch.equal(out[i][k][:c], want)
            assert (out[i][k][c:] == -7).all()
    ptr[0][0] = None
    with pytest.raises(ValueError):
        L.check(L.lib().tsc_pair_lists_each(tables[0].data_ptr(), tables[1].data_ptr(), K, cap,
                                            (ctypes.c_int64 * K)(*sizes), ptr[0], ptr[1],
                                            L.stream_of(tables)), "lists")
