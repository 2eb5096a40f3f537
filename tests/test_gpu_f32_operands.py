"""f32 layers whose operands lie at both ends of the exponent range: three
bf16 values hold an operand to 2^-134, which the other operand multiplies."""
import pytest
import torch

from gpu_util import DEV, needs_gpu, say
from test_gpu_conv import _conv_raw, _module, _tiny
from test_gpu_f32_split import _exact
from trispconv_amd import _lib as L
from trispconv_amd.pytorch.indices import generate_subm_indice_pairs
from trispconv_amd.pytorch.weight import pack_weight

pytestmark = [pytest.mark.gpu, needs_gpu]

# the slot-split kernel, the register-gather kernel (C_in = 48, and at 128
# columns), the direct-to-LDS kernel at 32 and at 64 rows per wave
LAYERS = [(64, 64, 3000, 24, 0), (48, 96, 30_000, 48, 0), (64, 128, 5000, 32, 128),
          (64, 64, 70_001, 64, 0), (64, 64, 270_007, 128, 0)]


def _layer(c_in, c_out, n, grid, f_scale, w_scale):
    idx = _tiny(23, (grid,) * 3, 1, n)
    data = generate_subm_indice_pairs(torch.from_numpy(idx).to(DEV), (grid,) * 3, 1, 3)
    g = torch.Generator().manual_seed(c_in + n)
    feats = (torch.randn(n, c_in, generator=g).double() * f_scale).float().to(DEV)
    m = _module("subm", c_in, c_out, 3, dtype=torch.float32, seed=9)
    with torch.no_grad():
        m.weight.copy_((m.weight.double() * w_scale).float())
        m.bias.zero_()
    say("f32 operands", c_in, c_out, n, f_scale, w_scale,
        L.lib().tsc_conv_kernel_name(L.F32, c_in, c_out, 27, n))
    return data.neighbour_map(n, DEV), feats, m


def _check(out, ref):
    """As in the split's own precision test: a random walk of 27 * C_in
    roundings of 2^-24, and the three products left out."""
    err = float((out.double() - ref).norm() / ref.norm())
    say("   rel err", err)
    assert err <= 1.2e-6 + 2.0 ** -24


@pytest.mark.parametrize("c_in,c_out,n,grid,tile", LAYERS)
@pytest.mark.parametrize("f_scale,w_scale", [
    (1e-36, 1e18), (2.4e-38, 1e18), (1e18, 1e-36),  # normal values on both sides
    (1e-43, 1e30), (1e30, 1e-43),                   # subnormal ones, which bf16 has no place for
    (1e-43, 1e37), (1.0, 1e30), (1e-20, 1e-14)])
def test_small_against_large_operands(c_in, c_out, n, grid, tile, f_scale, w_scale):
    nbr, feats, m = _layer(c_in, c_out, n, grid, f_scale, w_scale)
    out = _conv_raw(feats, m._packed_weight(torch.float32), m.bias, nbr, None, 0, n, tile)
    _check(out, _exact(feats, m, nbr))


@pytest.mark.parametrize("c_in,c_out,n,grid,tile", LAYERS)
def test_rows_of_small_values_among_ordinary_ones(c_in, c_out, n, grid, tile):
    """Every tenth row's features are subnormal, and a stretch of rows has
    none but zeros beside them: the rows that gather only such values are
    what float64 says, and all others keep the bits that they have in a layer
    without them (absent values add exact zeros)."""
    nbr, feats, m = _layer(c_in, c_out, n, grid, 1.0, 1e20)
    pw = m._packed_weight(torch.float32)
    small = torch.zeros(n, dtype=torch.bool, device=DEV)
    small[::10] = True
    lone = torch.zeros(n, dtype=torch.bool, device=DEV)
    lone[n // 4:n // 2] = True
    zeroed = torch.where(small[:, None] | lone[:, None], 0.0, feats)
    mixed = torch.where(small[:, None], feats * 1e-43, zeroed)
    a = _conv_raw(mixed, pw, m.bias, nbr, None, 0, n, tile)
    b = _conv_raw(zeroed, pw, m.bias, nbr, None, 0, n, tile)
    sees = lambda rows: ((nbr >= 0) & rows[nbr.clamp(min=0).long()]).any(0)  # noqa: E731
    ordinary = sees(~small & ~lone)
    only = ~ordinary & sees(small)
    assert int(only.sum()) > 10
    assert torch.equal(a[~ordinary & ~only], b[~ordinary & ~only])
    # 1e-43 * 1e20 is far below the last bit of an ordinary sum, but may turn one over
    assert torch.allclose(a[ordinary], b[ordinary], rtol=2.0 ** -22, atol=1e20 * 2.0 ** -22)
    keep = ordinary & ~sees(small)
    assert torch.equal(a[keep], b[keep])
    _check(a[only], _exact(mixed, m, nbr)[only])


@pytest.mark.parametrize("c_in,c_out", [(64, 64), (48, 96), (16, 32)])
@pytest.mark.parametrize("layout", ["krsc", "flat"])
def test_dead_columns_and_vanishing_rows(c_in, c_out, layout):
    """Columns without a weight stay zero while their rows' subnormal features
    count in the others; one column has its only weight in the last slot."""
    nbr, feats, m = _layer(c_in, c_out, 9000, 48, 1e-43, 1e30)
    n = len(feats)
    with torch.no_grad():
        m.weight[[0, 5, c_out - 1]] = 0
        m.weight[7] = 0
        m.weight[7, 2, 2, 2, c_in - 1] = 3e29
    w = m.weight.detach()
    pw = m._packed_weight(torch.float32)
    if layout == "flat":
        flat = w.reshape(c_out, 27, c_in).permute(1, 2, 0).contiguous()
        pw = pack_weight(flat, (27, 1, 1), c_in, c_out, torch.float32)
    out = _conv_raw(feats, pw, m.bias, nbr, None, 0, n, 0)
    ref = _exact(feats, m, nbr)
    assert (out[:, [0, 5, c_out - 1]] == 0).all()
    _check(out, ref)
    _check(out[:, 7], ref[:, 7])
    assert ((out == 0) == (ref == 0)).all()


def test_zero_weights_and_zero_rows_give_zeros():
    """Exact zeros stay zeros: dead columns, an all-zero weight, all-zero
    features, and rows without a pair of a wider map."""
    nbr, feats, m = _layer(64, 64, 30_000, 48, 1.0, 1.0)
    n = len(feats)
    with torch.no_grad():
        m.weight[5].zero_()
    out = _conv_raw(feats, m._packed_weight(torch.float32), m.bias, nbr, None, 0, n, 0)
    assert (out[:, 5] == 0).all()
    _check(out, _exact(feats, m, nbr))
    assert (_conv_raw(feats * 0, m._packed_weight(torch.float32), m.bias, nbr, None, 0, n, 0) == 0).all()
    empty = nbr.clone()
    empty[:, 100:300] = -1
    out = _conv_raw(feats, m._packed_weight(torch.float32), m.bias, empty, None, 0, n, 0)
    assert (out[100:300] == 0).all()
    with torch.no_grad():
        m.weight.zero_()
    assert (_conv_raw(feats, m._packed_weight(torch.float32), m.bias, nbr, None, 0, n, 0) == 0).all()
