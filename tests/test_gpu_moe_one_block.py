"""moe_create_indices in one block: around the edges of its waves and steps, of its limits and of the ids' range, equal to a
stable sort."""
import numpy as np
import pytest
import torch

import modular_amd as mx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("num_experts", [1, 3, 256, 511, 512, 513])
@pytest.mark.parametrize("n", [0, 1, 63, 64, 65, 513, 1023, 1024, 1025, 2048, 2049, 3333, 4095, 4096, 4097])
@pytest.mark.parametrize("kind", ["uniform", "one", "outside"])
def test_stable_sort(dev, n, num_experts, kind):
    rng = np.random.default_rng(n + 7 * num_experts)
    ids = rng.integers(0, num_experts, n).astype(np.int32)
    if kind == "one":
        ids[:] = num_experts - 1
    if kind == "outside":  # such assignments belong to no expert
        ids = rng.choice(np.array([-1, num_experts, num_experts + 512, -2**31, 0, num_experts - 1], dtype=np.int32), n)
    shifted = torch.from_numpy(np.concatenate([[0], ids]).astype(np.int32)).to(dev)[1:]  # 4-byte aligned
    order, start, restore, eids, stats = (t.cpu().view(torch.int32).numpy() for t in mx.moe_create_indices(shifted, num_experts))
    valid = np.flatnonzero((ids >= 0) & (ids < num_experts))
    counts = np.bincount(ids[valid], minlength=num_experts)
    want = valid[np.argsort(ids[valid], kind="stable")]
    assert np.array_equal(start, np.concatenate([[0], np.cumsum(counts)]))
    assert np.array_equal(order[:len(want)], want)
    assert np.array_equal(restore[want], np.arange(len(want)))
    assert np.array_equal(eids, np.arange(num_experts))
    assert stats[0] == (counts.max() if n else 0) and stats[1] == num_experts
