"""Row counts on both sides of each line of the 32x32-tile layers' kernel and
tile choice."""
import pytest
import torch

from gpu_util import DEV, needs_gpu, rel_err, say, to_np
from test_gpu_conv import TOL, _conv_raw, _module, _tiny
from trispconv_amd import _lib as L
from trispconv_amd.pytorch.indices import generate_subm_indice_pairs
from trispconv_amd.pytorch.weight import pack_weight

pytestmark = [pytest.mark.gpu, needs_gpu]


@pytest.mark.parametrize("c_in,c_out,dtype,rows", [
    (64, 64, torch.float16, (8192, 8193)),        # slot split / 32 columns
    (64, 32, torch.bfloat16, (32768, 32769)),     # the same, one column tile
    (64, 64, torch.float16, (22912, 22913)),      # 32 / 64 columns
    (128, 128, torch.bfloat16, (51072, 51073)),   # 64 / 128 columns
    (64, 64, torch.float16, (131072, 131073)),    # 32 / 64 rows per wave
    (128, 128, torch.float16, (98304, 98305)),
    (64, 64, torch.float32, (20480, 20481)),      # slot split / 32 columns
    (48, 64, torch.float32, (32768, 32769)),      # slot split / register gather
    (64, 64, torch.float32, (65408, 65409)),      # 32 / 64 columns
    (64, 64, torch.float32, (98304, 98305)),      # 32 / 64 rows per wave
    (48, 64, torch.float16, (20480, 20481)),      # slot split / register gather
    (48, 64, torch.float16, (32512, 32513)),      # 32 / 64 columns
    (48, 128, torch.bfloat16, (91904, 91905)),    # 64 / 128 columns
])
def test_own_choice_matches_the_forced_kernel(c_in, c_out, dtype, rows):
    """The layer's own choice against the register-gather kernel at 32 columns
    (itself against the oracle in the layer tests): the same bits, or, where
    the slot-split kernel sums in another order, within the layers'
    tolerance."""
    for n in rows:
        e = 96
        idx = _tiny(n, (e, e, e), 1, n)
        data = generate_subm_indice_pairs(torch.from_numpy(idx).to(DEV), (e, e, e), 1, 3)
        nbr = data.neighbour_map(n, DEV)
        g = torch.Generator().manual_seed(n)
        feats = torch.randn(n, c_in, generator=g).to(DEV).to(dtype)
        m = _module("subm", c_in, c_out, 3, dtype=dtype, seed=3)
        pw = m._packed_weight(dtype)
        name = L.lib().tsc_conv_kernel_name(L.dtype_code(dtype), c_in, c_out, 27, n)
        say("tile choice", c_in, c_out, dtype, n, name)
        own = _conv_raw(feats, pw, m.bias, nbr, None, 0, n, 0)
        ref = _conv_raw(feats, pw, m.bias, nbr, None, 0, n, 32)
        if name == b"conv_split_kernel":
            assert rel_err(to_np(own), to_np(ref)) <= TOL[dtype]
        else:
            assert torch.equal(own, ref)


@pytest.mark.parametrize("c_in,c_out,K,dtype,split,n", [
    # strided and inverse layers: the slot split goes further
    (64, 64, 27, torch.float16, True, 16384), (64, 64, 27, torch.float16, False, 16385),
    (64, 64, 8, torch.bfloat16, True, 16384), (64, 64, 8, torch.bfloat16, False, 16385),
    (48, 64, 8, torch.float16, True, 16384), (48, 64, 8, torch.float16, False, 16385),
    (48, 64, 27, torch.float16, True, 20480), (48, 64, 27, torch.float16, False, 20481),
    (64, 64, 27, torch.float32, True, 32768), (64, 64, 27, torch.float32, False, 32769),
    (64, 32, 27, torch.float32, True, 40960), (64, 32, 27, torch.float32, False, 40961),
    # short slot lists: no split, tiles by 512 256-row ones
    (64, 64, 3, torch.float32, False, 900), (64, 64, 3, torch.float16, False, 131_073),
    # 64 rows per wave where 256-row tiles fit the chip at once, but not with
    # fewer input than output rows
    (128, 128, 27, torch.bfloat16, False, 100_000),
    (64, 64, 27, torch.float32, False, 100_000)])
@pytest.mark.parametrize("n_in", ["fewer", "more"])
def test_layers_of_other_input_than_output_rows(c_in, c_out, K, dtype, split, n, n_in):
    """The same on both sides of the lines that such layers have, over maps of
    rows that use an eighth to all of the slots."""
    rows = max(n // 4, 1) if n_in == "fewer" else n + n // 2
    g = torch.Generator().manual_seed(n)
    nbr = torch.randint(0, rows, (K, n), generator=g, dtype=torch.int32)
    use = torch.rand(K, n, generator=g) < torch.rand(n, generator=g) * 0.9 + 0.1
    nbr = torch.where(use, nbr, -1).to(DEV)
    feats = torch.randn(rows, c_in, generator=g).to(DEV).to(dtype)
    w = (torch.randn(K, c_in, c_out, generator=g) / (K * c_in) ** 0.5).to(DEV).to(dtype)
    bias = torch.randn(c_out, generator=g).to(DEV).to(dtype)
    pw = pack_weight(w, (K, 1, 1), c_in, c_out, dtype)
    own = _conv_raw(feats, pw, bias, nbr, None, 0, n, 0)
    ref = _conv_raw(feats, pw, bias, nbr, None, 0, n, 32)
    say("tile choice", c_in, c_out, K, dtype, rows, "->", n, "same bits", torch.equal(own, ref))
    assert rel_err(to_np(own), to_np(ref)) <= TOL[dtype]
    # the split's four partial sums round otherwise somewhere in thousands of outputs
    assert torch.equal(own, ref) == (not split)
