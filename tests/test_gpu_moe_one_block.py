"""moe_create_indices in one block: around the edges of its waves and steps, of its limits and of the ids' range, equal to a
stable sort."""
import numpy as np
import pytest
import torch

import modular_amd as mx
from modular_amd import _lib, synth
from util import assert_rel, f32_np

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


@pytest.mark.parametrize("n", [700, 4096, 6000])
def test_assignments_without_an_expert_have_no_position(dev, n):
    """... whatever the buffer held: left as it was, it would be read as a position and another assignment's row overwritten."""
    ids = torch.randint(-2, 12, (n,), generator=torch.Generator().manual_seed(n)).to(torch.int32).to(dev)
    buf = lambda size: torch.zeros((size,), dtype=torch.int32, device=dev)
    order, start, restore, eids, stats = buf(n), buf(11), buf(n), buf(10), buf(2)
    lib = _lib.lib()
    for at in (ids, torch.cat([ids[:1], ids])[1:]):   # 16-byte and 4-byte aligned
        restore.zero_()
        _lib.check(lib.maxfp8_moe_create_indices(order.data_ptr(), start.data_ptr(), restore.data_ptr(), eids.data_ptr(), stats.data_ptr(),
                                                    at.data_ptr(), n, 10, torch.cuda.current_stream().cuda_stream))
        valid = (ids >= 0) & (ids < 10)
        assert (restore[~valid] == -1).all()
        assert torch.equal(torch.sort(restore[valid]).values, torch.arange(int(valid.sum()), dtype=torch.int32, device=dev))


@pytest.mark.parametrize("seq,host_sync", [(40, False), (40, True), (1500, True)])
def test_experts_of_ids_out_of_range(dev, seq, host_sync):
    """The assignments to an expert get the rows they get with every id in range (other rows in their tiles: the order of a
    tile kind's sums may differ, not more)."""
    E, k, H, F = 6, 3, 256, 128
    cfg = mx.blockwise_fp8_config()
    weight = lambda n, kk, seed: tuple(torch.stack(t).to(dev) for t in zip(*[
        synth.quantize_weight_block(synth.weights_f32(n, kk, seed=seed + e)) for e in range(E)]))
    (gu, sgu), (d, sd) = weight(2 * F, H, 1), weight(H, F, 50)
    x = synth.activations(seq, H, seed=3, device=dev)
    g = torch.Generator().manual_seed(4)
    router = torch.randn((seq, E), generator=g).topk(k, dim=1).indices.to(torch.int32)
    want = mx.expert_matmuls_fp8(x, router.to(dev), gu, sgu, d, sd, cfg, host_sync=host_sync)
    gone = torch.rand((seq, k), generator=g) < 0.3
    router[gone] = torch.tensor([-1, E, 2**31 - 1], dtype=torch.int32)[torch.randint(0, 3, (int(gone.sum()),), generator=g)]
    for _ in range(3):                                 # (over buffers of the call before)
        got = mx.expert_matmuls_fp8(x, router.to(dev), gu, sgu, d, sd, cfg, host_sync=host_sync)
        assert_rel(f32_np(got[~gone]), f32_np(want[~gone]), 1e-2, "experts with ids out of range")
    nobody = torch.full((seq, k), -1, dtype=torch.int32, device=dev)
    assert mx.expert_matmuls_fp8(x, nobody, gu, sgu, d, sd, cfg, host_sync=host_sync).shape == (seq, k, H)
    torch.cuda.synchronize()
