"""The records commit over its tilings: value dims off the row tile, every key dim, paths longer than a staged strip (16
nodes) and tables wider than a wave, records on any 4-byte boundary, against the oracle (fp32 states 1e-4, 16-bit pools
1e-2, as the commit's other tests)."""

import pytest
import torch

from conftest import announce, assert_states_close
from oracle import records as orec

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,layers,n,pool_dtype,spare,width", [
    ((128, 128), 6, 8, torch.bfloat16, 4, 40), ((128, 72), 2, 3, torch.float32, 1, 24), ((128, 200), 5, 30, torch.float16, 2, 17),
    ((64, 64), 5, 60, torch.float32, 3, 33), ((256, 96), 1, 3, torch.bfloat16, 1, 20), ((32, 40), 1, 3, torch.bfloat16, 1, 18),
    ((16, 16), 1, 2, torch.float32, 1, 16), ((8, 24), 1, 2, torch.float16, 1, 5), ((128, 64), 1, 2, torch.float32, 4, 80)])
def test_commit_tilings(dev, dims, layers, n, pool_dtype, spare, width):
    from eagle_harness.kernels.gdn_tree_records import gdn_tree_records_commit

    (K, V), HV = dims, 2
    announce(f"records commit K={K} V={V} layers={layers} n={n} {pool_dtype} width={width}")
    gen = torch.Generator().manual_seed(K + V + n)
    parent = torch.stack([torch.tensor([-1] + [j - 1 if i % 2 else int(torch.randint(0, j, (1,), generator=gen))
                                               for j in range(1, width)]) for i in range(n)])
    state = (torch.randn(layers, n + 1, HV, V, K, generator=gen) * 0.1).to(pool_dtype)
    records = torch.randn(layers, n, width, HV, V + K + spare, generator=gen) * 0.1
    records[..., V + K] = torch.rand(layers, n, width, HV, generator=gen) * 0.5 + 0.5
    slots = torch.arange(1, n + 1, dtype=torch.int32)
    steps = torch.tensor([min(width, 64) - 1 - i % 3 for i in range(n)], dtype=torch.int64)  # chains of up to 64 nodes
    if width > 64:
        parent[0, width - 1], steps[0] = 70, width - 1  # node 79 <- 70 <- 3: entries past a wave
        parent[0, 70], parent[0, 3] = 3, 0
    rounded = pool_dtype != torch.float32
    want = state.clone()
    orec.gdn_tree_records_commit(want, records, slots, torch.arange(n), steps, parent, rounded)
    got = state.to(dev)
    gdn_tree_records_commit(got, records.to(dev), slots.to(dev), torch.arange(n, device=dev), steps.to(dev), parent.to(dev),
                            rounded)
    if rounded:
        torch.testing.assert_close(got.cpu().float(), want.float(), atol=1e-2, rtol=1e-2)
    else:
        assert_states_close(got.cpu(), want)


@pytest.mark.parametrize("pool_dtype", [torch.bfloat16, torch.float32])
def test_skipped_requests_have_no_parents(dev, pool_dtype):
    """A batch padded past its parent table's rows: the padding is skipped (a negative step, slot or row) or accepted at
    its root, which has no parent, and none of that reads the table."""
    from eagle_harness.kernels.gdn_tree_records import gdn_tree_records_commit

    announce(f"records commit, padded batch {pool_dtype}")
    gen = torch.Generator().manual_seed(3)
    layers, n, width, HV, V, K = 2, 6, 9, 2, 64, 128
    parent = torch.tensor([[-1, 0, 1, 2, 3, 4, 5, 6, 7], [-1, 0, 0, 1, 1, 2, 2, 3, 3]])
    state = (torch.randn(layers, n + 1, HV, V, K, generator=gen) * 0.1).to(pool_dtype)
    records = torch.randn(layers, n, width, HV, V + K + 1, generator=gen) * 0.1
    slots, rows = torch.tensor([1, 2, 3, -1, 5, 6]), torch.tensor([0, 1, 2, 3, -1, 5])
    steps = torch.tensor([8, 7, -1, 4, 4, 0])
    rounded = pool_dtype != torch.float32
    want = state.clone()
    orec.gdn_tree_records_commit(want, records, slots, rows, steps, parent, rounded)
    got = state.to(dev)
    gdn_tree_records_commit(got, records.to(dev), slots.to(dev), rows.to(dev), steps.to(dev), parent.to(dev), rounded)
    if rounded:
        torch.testing.assert_close(got.cpu().float(), want.float(), atol=1e-2, rtol=1e-2)
    else:
        assert_states_close(got.cpu(), want)
    assert torch.equal(got.cpu()[:, [0, 3, 4, 5]], state[:, [0, 3, 4, 5]])
