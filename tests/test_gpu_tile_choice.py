"""Row counts on both sides of each line of the 32x32-tile layers' kernel and
tile choice."""
import pytest
import torch

from gpu_util import DEV, needs_gpu, rel_err, say, to_np
from test_gpu_conv import TOL, _conv_raw, _module, _tiny
from trispconv_amd import _lib as L
from trispconv_amd.pytorch.indices import generate_subm_indice_pairs

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
