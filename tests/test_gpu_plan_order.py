"""The execution order against the sort it stands for, made on the host."""
import numpy as np
import pytest
import torch

from gpu_util import DEV, needs_gpu, say
from trispconv_amd import _lib as L

pytestmark = [pytest.mark.gpu, needs_gpu]

TILE = 256


def _order(masks, region):
    """Columns sorted by (region, slot mask), ties as they come; then each
    region's whole tiles by the slots that their rows use, most first."""
    n = len(masks)
    at = np.lexsort((np.arange(n), masks, np.arange(n) // region))
    full = n // TILE
    union = np.bitwise_or.reduce(masks[at[:full * TILE]].reshape(full, TILE), axis=1)
    slots = np.array([bin(int(u)).count("1") for u in union])
    tiles = np.lexsort((np.arange(full), -slots, np.arange(full) // max(region // TILE, 1)))
    return np.concatenate([at[:full * TILE].reshape(full, TILE)[tiles].ravel(), at[full * TILE:]])


def _masks(kind, n, K, rng):
    """Slot masks as scenes have them: `lead` sizes of buckets that share their
    leading nine bits; one layer of voxels (the planes above and below empty,
    so every row shares them); all alike; anything."""
    if kind == "plane":
        return rng.integers(1, 512, n) << min(9, K - 9) if K > 9 else rng.integers(1, 1 << K, n)
    if kind == "alike":
        return np.full(n, (1 << K) - 1)
    if kind == "any":
        return rng.integers(0, 1 << K, n)
    low = K - 9
    lead = rng.permutation(np.repeat(np.arange(len(kind)) * 37 % 512, kind))[:n]
    return (lead << low) | rng.integers(0, 1 << low, n)


@pytest.mark.parametrize("K,kind,n", [
    (27, "any", 1), (27, "any", 255), (27, "any", 256), (27, "any", 5121), (27, "any", 60_000),
    (27, [5119, 5120, 5121, 10241, 300], 25_901), (10, [5120, 5121, 9000], 19_241),
    (27, "plane", 5120), (27, "plane", 40_003), (27, "alike", 30_000),
    (12, "any", 20_000), (28, "any", 20_000), (28, [17_000, 100, 20], 17_120), (29, "any", 7000),
    (32, "any", 20_000), (9, "any", 9000), (1, "any", 3000)])
@pytest.mark.parametrize("region", [1 << 30, 8192])
def test_order_is_the_stable_sort_by_mask(K, kind, n, region):
    rng = np.random.default_rng(n + K)
    masks = _masks(kind, n, K, rng).astype(np.int64)
    say("plan order", K, kind, n, region, "distinct masks", len(np.unique(masks)))
    bits = ((masks[None] >> np.arange(K)[:, None]) & 1).astype(bool)
    nbr = np.where(bits, rng.integers(0, n, (K, n)), -1).astype(np.int32)
    nbr_d = torch.from_numpy(nbr).to(DEV)
    lib = L.lib()
    ws = L.workspace(lib.tsc_plan_workspace_bytes(n, K), nbr_d.device)
    order = torch.empty(n, dtype=torch.int32, device=DEV)
    ordered = torch.empty((K, n), dtype=torch.int32, device=DEV)
    pos_masks = torch.empty(n, dtype=torch.int32, device=DEV)
    L.check(lib.tsc_conv_plan(nbr_d.data_ptr(), None, 1, None, n, K, 1, L.i3((64, 64, 64)), region,
                              ws.data_ptr(), ws.numel(), order.data_ptr(), ordered.data_ptr(),
                              pos_masks.data_ptr(), L.stream_of(nbr_d)), "plan")
    want = _order(masks, min(region, max(n, 1)))
    got = order.cpu().numpy()
    assert np.array_equal(np.sort(got), np.arange(n))
    assert np.array_equal(got, want)
    assert np.array_equal(ordered.cpu().numpy(), nbr[:, want])
    assert np.array_equal(pos_masks.cpu().numpy().astype(np.uint32).astype(np.int64), masks[want])
