"""Where an inverse's columns are grouped: by the matrix work of the layer that
asks first, on both sides of the line."""
import pytest
import torch

from trispconv_amd.pytorch import indices as I


@pytest.mark.parametrize("c_in,c_out,k,dtype,below,above", [
    (64, 32, 3, torch.bfloat16, 180_000, 182_000), (128, 64, 3, torch.float16, 45_000, 45_500),
    (64, 32, 3, torch.float32, 45_000, 45_500), (128, 64, 2, torch.bfloat16, 152_000, 153_000)])
def test_the_line(c_in, c_out, k, dtype, below, above, monkeypatch):
    e = torch.empty(0, 4, dtype=torch.int32)
    got = []
    monkeypatch.setattr(I, "_inverse_pairs", lambda fwd, work: got.append(work))

    def fwd(stride):
        d = I.IndiceData(e, None, None, None, e, (64,) * 3, (32,) * 3, (k,) * 3, (stride,) * 3, (0,) * 3,
                         (1,) * 3, False)
        d._geo = ((k,) * 3, (stride,) * 3, (0,) * 3, (1,) * 3)
        return d
    I.inverse_pairs_for(fwd(2), c_in, c_out, dtype)
    assert not I._group_inverse(fwd(2), below, got[0])
    assert I._group_inverse(fwd(2), above, got[0])
    assert not I._group_inverse(fwd(1), above, got[0])   # one residue class
    assert not I._group_inverse(fwd(5), above, got[0])   # 125 of them
    I.inverse_pairs_for(fwd(2), c_in, 20, dtype)         # a layer that runs every slot anyway
    assert not I._group_inverse(fwd(2), 1 << 30, got[1])
    made = fwd(2)
    made._geo = None                                      # not built here
    assert not I._group_inverse(made, above, got[0])
