"""The snapshot walk with 32 staged nodes against 16 (the requests' mean rows choose, at most the per-row slot table's
columns): trees around both counts, in both lane forms and pool dtypes, bit for bit the same under either count, and
against the oracle."""

import numpy as np
import pytest
import torch

from conftest import announce, assert_states_close
from oracle import recurrence as orr
from workloads import seeded_tree

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("value_heads,n", [(2, 5), (24, 11)])  # the small grids' form, and the 8-lane form
@pytest.mark.parametrize("pool_dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("in_dtype", [torch.bfloat16, torch.float32])
def test_staged_counts_agree(dev, value_heads, n, pool_dtype, in_dtype):
    from eagle_harness.kernels.gdn_tree_recurrence import gdn_tree_recurrent_update

    announce(f"walk staging heads={value_heads} {pool_dtype} {in_dtype}")
    rng, gen = np.random.default_rng(n), torch.Generator().manual_seed(n)
    sizes = ([16, 17, 31, 32, 33, 40, 1, 64, 18, 24, 15])[:n]
    H, K, V, width = 2, 128, 32, 64
    tokens = sum(sizes)
    cu = torch.tensor([0] + np.cumsum(sizes).tolist(), dtype=torch.int32)
    parents = torch.full((n, width), -1, dtype=torch.int32)
    for i, size in enumerate(sizes):
        parents[i, :size] = torch.tensor(seeded_tree(rng, size), dtype=torch.int32)
    rnd = lambda *s: torch.randn(*s, generator=gen)  # noqa: E731
    q, k, v = rnd(1, tokens, H, K).to(in_dtype), rnd(1, tokens, H, K).to(in_dtype), rnd(1, tokens, value_heads, V).to(in_dtype)
    a, b = rnd(tokens, value_heads).bfloat16(), rnd(tokens, value_heads).bfloat16()
    A_log, dt_bias = torch.zeros(value_heads), torch.zeros(value_heads)
    slots = (1 + torch.randperm(n * width, generator=gen)).to(torch.int32).view(n, width)
    pool = torch.zeros(1 + n * width, value_heads, V, K, dtype=pool_dtype)
    pool[slots[:, 0].long()] = (rnd(n, value_heads, V, K) * 0.1).to(pool_dtype)

    def run(fn, d, table, p, publish=None):
        out = torch.zeros_like(v).to(d)
        fn(A_log.to(d), dt_bias.to(d), q.to(d), k.to(d), v.to(d), a.to(d), b.to(d), initial_state_source=p,
           initial_state_indices=table, cu_seqlens=cu.to(d), intermediate_states_buffer=p, intermediate_state_indices=table,
           retrieve_parent_token=parents.to(d), num_accepted_tokens=torch.ones(n, dtype=torch.int32, device=d), pad_slot_id=0,
           out=out)
        return out.cpu(), p.cpu()

    table = slots.to(dev)
    wide_out, wide_pool = run(gdn_tree_recurrent_update, dev, table, pool.clone().to(dev))
    # the same slots under a table that names 16 columns: its rows keep their stride, so later columns are still there
    narrow_out, narrow_pool = run(gdn_tree_recurrent_update, dev, table[:, :16], pool.clone().to(dev))
    # a node's norms are summed in one order whether it is staged or loaded in the walk: not a bit differs
    assert torch.equal(wide_pool, narrow_pool)
    assert torch.equal(wide_out, narrow_out)
    want_pool = pool.clone()
    want, want_pool = run(orr.gdn_tree_recurrent_update, torch.device("cpu"), slots, want_pool)
    tol = dict(atol=1e-4, rtol=1e-4) if in_dtype == pool_dtype == torch.float32 else dict(atol=2e-2, rtol=2e-2)
    torch.testing.assert_close(wide_out.float(), want.float(), **tol)
    if pool_dtype == torch.float32:
        assert_states_close(wide_pool, want_pool)
    else:
        torch.testing.assert_close(wide_pool.float(), want_pool.float(), atol=1e-2, rtol=1e-2)
