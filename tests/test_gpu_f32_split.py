"""f32 layers on the bf16 matrix cores (each operand a sum of three bf16
values): precision, and values that no such sum holds."""
import numpy as np
import pytest
import torch

from gpu_util import DEV, needs_gpu, say
from test_gpu_conv import _conv_raw, _module, _tiny
from trispconv_amd import _lib as L
from trispconv_amd.pytorch.indices import generate_subm_indice_pairs

pytestmark = [pytest.mark.gpu, needs_gpu]


def _exact(feats, m, nbr):
    """The layer in float64 on the GPU, slot by slot."""
    w = m.weight.detach().double()
    w = w.reshape(w.shape[0], -1, w.shape[-1]).permute(1, 2, 0).contiguous()
    out = m.bias.detach().double().expand(nbr.shape[1], -1).clone()
    f = feats.double()
    for k in range(nbr.shape[0]):
        rows = (nbr[k] >= 0).nonzero()[:, 0]
        out[rows] += f[nbr[k][rows].long()] @ w[k]
    return out


# the slot-split kernel (rows of one partial tile and of several), the
# register-gather kernel (C_in = 48), the direct-to-LDS kernel at 32 and at 64
# rows per wave
@pytest.mark.parametrize("c_in,c_out,n,grid,tile", [(48, 64, 20_000, 40, 0), (64, 64, 50, 12, 0),
                                                    (48, 32, 3000, 24, 0), (64, 64, 150_001, 96, 0),
                                                    (64, 64, 300_007, 128, 0), (32, 32, 30_000, 64, 0),
                                                    (64, 128, 5000, 32, 128)])
@pytest.mark.parametrize("scale", [1.0, 1e-12, 1e15, 1e-34])
def test_split_precision_and_non_finite_rows(c_in, c_out, n, grid, tile, scale):
    """Against float64: at most 27 * C_in products summed in f32, so a random
    walk of that many roundings of 2^-24 bounds the relative 2-norm error
    (sqrt(27 * 64) * 2^-25 = 1.2e-6; the three products left out add below
    2^-24).  Then rows of +inf, NaN and the largest f32 value are planted: the
    outputs without such a neighbour keep their bits, the others are what
    float64 says where that is not finite."""
    idx = _tiny(17, (grid, grid, grid), 1, n)
    data = generate_subm_indice_pairs(torch.from_numpy(idx).to(DEV), (grid,) * 3, 1, 3)
    nbr = data.neighbour_map(n, DEV)
    g = torch.Generator().manual_seed(c_in + n)
    feats = (torch.randn(n, c_in, generator=g) * scale).to(DEV)
    m = _module("subm", c_in, c_out, 3, dtype=torch.float32, seed=5)
    with torch.no_grad():
        m.bias.mul_(scale)
    pw = m._packed_weight(torch.float32)
    say("f32 split", c_in, c_out, n, scale, L.lib().tsc_conv_kernel_name(L.F32, c_in, c_out, 27, n))
    out = _conv_raw(feats, pw, m.bias, nbr, None, 0, n, tile)
    ref = _exact(feats, m, nbr)
    err = float((out.double() - ref).norm() / ref.norm())
    say("   rel err", err)
    assert err <= 1.2e-6 + 2.0 ** -24
    bad = feats.clone()
    rows = torch.tensor([3, n // 2, n - 1], device=DEV)
    bad[rows] = torch.tensor([[float("inf")], [float("nan")], [3.4028235e38]], device=DEV)
    got = _conv_raw(bad, pw, m.bias, nbr, None, 0, n, tile)
    ref = _exact(bad, m, nbr).float()
    touched = (nbr.unsqueeze(-1) == rows).any(-1).any(0)
    assert torch.equal(got[~touched], out[~touched])
    assert int(touched.sum()) >= 3
    a, b = got[touched], ref[touched]
    # beside the largest finite value a sum may pass infinity on its way
    near = (nbr == n - 1).any(0)[touched]
    assert torch.equal(torch.isnan(a[~near]), torch.isnan(b[~near]))
    inf = torch.isinf(b) & ~near[:, None]
    assert torch.equal(a[inf], b[inf])
    own = (nbr == n - 1).any(0) & ~((nbr == 3) | (nbr == n // 2)).any(0)
    fin = own[:, None] & torch.isfinite(ref) & (ref.abs() < 1e38)
    # such a sum cancels: C_in products of up to big * max|w| each, summed with a
    # rounding of 2^-24 of at most their absolute sum at each of C_in steps
    # (the other neighbours' products are far below)
    bound = c_in * c_in * 2.0 ** -24 * 3.4028235e38 * float(m.weight.abs().max())
    assert float((got[fin].double() - ref[fin].double()).abs().max()) <= bound
