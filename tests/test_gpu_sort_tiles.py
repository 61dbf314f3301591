"""Stable sorts on both sides of the sizes where the number of keys per thread changes (2^18 and 2^19), and of the
edges of the tiles of 1,024 and 2,048 keys, against numpy's stable sort (exact)."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1023, 1024, 1025, (1 << 18) - 1, 1 << 18, (1 << 18) + 1, (1 << 19) - 1, 1 << 19, (1 << 19) + 1])
@pytest.mark.parametrize("bits", [30, 64])
def test_sort_around_tile_rules(gwn, dev, n, bits):
    import torch

    rng = np.random.default_rng(n)
    # Few different keys: runs of equal ones cross tiles, so a lost order of tiles shows.
    word, view = (np.uint32, np.int32) if bits == 30 else (np.uint64, np.int64)
    keys = rng.choice(rng.integers(0, 1 << (bits - 1), size=5000, dtype=np.uint64).astype(word), size=n)
    dk = torch.from_numpy(keys.view(view)).to(dev)
    dv = torch.from_numpy(np.arange(n, dtype=np.int32)).to(dev)
    gwn.radix_sort_pairs(dk, dv, 0, bits).raise_if_error()
    torch.cuda.synchronize()
    order = np.argsort(keys, kind="stable")
    assert np.array_equal(dv.cpu().numpy(), order.astype(np.int32))
    assert np.array_equal(dk.cpu().numpy().view(word), keys[order])
