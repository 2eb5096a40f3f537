"""Widths that fill no whole pieces or tiles, with weights of another type than
the 16-bit features they are packed for: the weights keep their own values."""
import numpy as np
import pytest
import torch

from gpu_util import DEV, needs_gpu, say
from test_gpu_conv import _conv_raw, _tiny
from trispconv_amd import _lib as L
from trispconv_amd.pytorch import functional as F
from trispconv_amd.pytorch.indices import generate_subm_indice_pairs
from trispconv_amd.pytorch.weight import pack_weight

pytestmark = [pytest.mark.gpu, needs_gpu]

HALF_ULP = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}


def _exact(f, w, b, nbr):
    """(the layer, the sums of its products' magnitudes) in float64."""
    out = b.double().expand(nbr.shape[1], -1).clone()
    mag = out.abs()
    f, w = f.double(), w.double()
    for k in range(len(nbr)):
        rows = (nbr[k] >= 0).nonzero()[:, 0]
        g = f[nbr[k][rows].long()]
        out[rows] += g @ w[k]
        mag[rows] += g.abs() @ w[k].abs()
    return out, mag


@pytest.mark.parametrize("dtype,w_dtype", [(torch.float16, torch.float32), (torch.bfloat16, torch.float32),
                                           (torch.float16, torch.bfloat16), (torch.bfloat16, torch.float16)])
@pytest.mark.parametrize("c_in,c_out,k,n", [(3, 16, 3, 3001), (5, 20, 3, 777), (16, 20, 3, 5000), (1, 16, 5, 900),
                                            (2, 32, 3, 1025), (4, 3, 3, 64), (96, 20, 1, 4000), (1, 1, 1, 1),
                                            (1, 7, 3, 2), (130, 65, 1, 333)])
def test_weights_keep_their_type(c_in, c_out, k, n, dtype, w_dtype):
    """Weights around 1 + 2^-9 a with features that cancel their ones (channel
    pairs, or the whole sum's leading part), and weights past both ends of
    f16's range: products in f32, so an error of at most C_in * K roundings of
    2^-24 of the summed magnitudes, and the result's own rounding."""
    rng = np.random.default_rng(n)
    e = max(4, int(np.ceil((3 * n) ** (1 / 3))))
    idx = _tiny(n, (e, e, e), 1, n)
    nbr = generate_subm_indice_pairs(torch.from_numpy(idx).to(DEV), (e,) * 3, 1, k).neighbour_map(n, DEV)
    K = k ** 3
    f = rng.standard_normal((n, c_in))
    f[:, 1::2] = -f[:, :c_in - c_in % 2:2]
    f = torch.from_numpy(f).to(DEV).to(dtype)
    near_one = 1 + rng.standard_normal((K, c_in, c_out)) * 2.0 ** -9
    wide = rng.standard_normal((K, c_in, c_out)) * rng.choice([1e-9, 3e5 if w_dtype != torch.float16 else 3e4],
                                                              (K, 1, c_out))
    b = torch.randn(c_out, device=DEV)
    for w in (near_one, wide):
        w = torch.from_numpy(w).to(DEV).to(w_dtype)
        say("ragged weights", c_in, c_out, k, n, dtype, w_dtype)
        pw = pack_weight(w, (k, k, k), c_in, c_out, dtype)
        out = _conv_raw(f, pw, b, nbr, None, 0, n, 0)
        ref, mag = _exact(f, w, b, nbr)
        bound = HALF_ULP[dtype] * ref.abs() + K * c_in * 2.0 ** -24 * mag + 2.0 ** -24
        top = torch.finfo(dtype).max
        fits = ref.abs() < top * 0.99
        assert ((out.double() - ref).abs() <= bound)[fits].all()
        assert torch.isinf(out[ref.abs() > top * 1.01]).all()


def test_packing_again_for_the_features_own_type_and_nan_weights():
    """One buffer for both forms, in turn; a NaN weight whatever its bits."""
    nbr = generate_subm_indice_pairs(torch.from_numpy(_tiny(1, (9, 9, 9), 1, 200)).to(DEV), (9,) * 3, 1,
                                     3).neighbour_map(200, DEV)
    f = torch.randn(200, 3, device=DEV).half()
    b = torch.zeros(16, device=DEV)
    w = torch.randn(27, 3, 16, device=DEV)
    half = pack_weight(w.half(), (3, 3, 3), 3, 16, torch.float16)
    full = pack_weight(w, (3, 3, 3), 3, 16, torch.float16)
    same = pack_weight(w.half().float(), (3, 3, 3), 3, 16, torch.float16)
    assert half.data.numel() == full.data.numel()
    run = lambda pw: _conv_raw(f, pw, b, nbr, None, 0, 200, 0)  # noqa: E731
    assert (run(same).float() - run(half).float()).abs().max() <= 2.0 ** -10 * run(half).float().abs().max()
    assert not torch.equal(run(full), run(half))
    lib = L.lib()
    for src in (w, w.half(), w):
        src = src.contiguous()
        L.check(lib.tsc_pack_weight(src.data_ptr(), L.dtype_code(src.dtype), 1, 27, 3, 16, L.F16,
                                    half.data.data_ptr(), L.stream_of(src)), "pack")
        want = full if src.dtype == torch.float32 else pack_weight(src, (3, 3, 3), 3, 16, torch.float16)
        assert torch.equal(run(half), run(want))
    bits = w.clone().view(torch.int32)
    bits[26, 2, 15] = 0x7fc5a51e  # the last weight of the f32 form
    out = run(pack_weight(bits.view(torch.float32), (3, 3, 3), 3, 16, torch.float16))
    uses = (nbr[26] >= 0)
    assert torch.isnan(out[uses, 15]).all() and torch.equal(out[~uses], run(full)[~uses])
    assert torch.equal(out[:, :15], run(full)[:, :15])


def test_through_the_layer_call():
    """sparse_conv_forward with such a packed weight: as the fp32 layer on the
    same values, rounded once."""
    n = 3000
    idx = torch.from_numpy(_tiny(4, (24, 24, 24), 1, n)).to(DEV)
    data = generate_subm_indice_pairs(idx, (24,) * 3, 1, 3)
    f, w, b = torch.randn(n, 5, device=DEV).half(), torch.randn(27, 5, 20, device=DEV), torch.randn(20, device=DEV)
    out = F.sparse_conv_forward(f, pack_weight(w, (3, 3, 3), 5, 20, torch.float16), b, data, n)
    ref = F.sparse_conv_forward(f, w, b, data, n)  # on fp32 copies
    err = (out.float() - ref.float()).abs()
    assert (err <= 2.0 ** -10 * ref.float().abs() + 1e-5).all()
