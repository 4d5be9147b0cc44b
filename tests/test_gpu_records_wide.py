"""The chunk form of trees of 17 to 64 nodes on the matrix cores: tile edges, rows in any order, every pool dtype,
against the oracle's closed form (fp32 records within 1e-4, as the narrower trees'), and values that are not finite,
which reach the node they are given to and its descendants only."""

import numpy as np
import pytest
import torch

from conftest import announce
from test_gpu_records import _call, _chunk_case, _inputs, _relabelled_tree, _to
from workloads import seeded_tree

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("width,dims,pool_dtype", [
    (17, (2, 4, 128, 128), torch.float32), (31, (1, 3, 64, 48), torch.bfloat16), (32, (2, 2, 128, 32), torch.float16),
    (33, (1, 2, 32, 16), torch.float32), (48, (2, 4, 128, 64), torch.bfloat16), (49, (1, 2, 64, 32), torch.float32),
    (64, (2, 4, 128, 128), torch.float32), (64, (1, 2, 128, 32), torch.float16)])
def test_wide_trees_match_the_closed_form(dev, width, dims, pool_dtype):
    announce(f"records chunk form width {width} dims={dims} pool={pool_dtype}")
    rng = np.random.default_rng(width)
    trees = [seeded_tree(rng, width), _relabelled_tree(rng, width), list(range(-1, width - 1)), [-1], [],
             seeded_tree(rng, 16), _relabelled_tree(rng, width - 1), seeded_tree(rng, width - 2)]

    def edit(inp):
        inp["state_indices"][6] = -1  # no pool slot: zeros
        inp["record_indices"][7] = -1  # outputs only

    _chunk_case(dev, trees, dims, pool_dtype, width, edit)


@pytest.mark.parametrize("width", [24, 40, 64])
@pytest.mark.parametrize("pool_dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_two_column_tiles_a_wave(dev, width, pool_dtype):
    """16 requests of 16 value heads and V 64: 512 waves of two column tiles, from where on a wave takes two."""
    announce(f"records chunk form width {width}, two column tiles, pool={pool_dtype}")
    rng = np.random.default_rng(width)
    trees = [(_relabelled_tree if i % 3 == 1 else seeded_tree)(rng, int(rng.integers(max(2, width - 20), width + 1)))
             for i in range(14)] + [list(range(-1, width - 1)), []]

    def edit(inp):
        inp["state_indices"][3] = -1  # no pool slot: zeros
        inp["record_indices"][4] = -1  # outputs only

    _chunk_case(dev, trees, (4, 16, 128, 64), pool_dtype, width + 1, edit)


@pytest.mark.parametrize("n,H,HV,V", [(1, 1, 2, 32), (16, 2, 16, 64)])  # one and two column tiles a wave
@pytest.mark.parametrize("what", ["v", "k", "a"])
def test_values_that_are_not_finite_stay_on_their_path(dev, what, n, H, HV, V):
    """One node's value, key or gate not finite: the node and its descendants get outputs that are not finite in the
    columns concerned, every other output keeps its bits."""
    from eagle_harness.kernels.gdn_tree_records import gdn_tree_chunk_update

    announce(f"records chunk form, {what} not finite")
    tree = [-1, 0, 1, 2, 0, 4, 5] + list(range(6, 30)) + [0, 31, 32]  # node 3's chain ends; 4 .. 30 one chain; 31 .. 33
    inp, width = _inputs([tree] * n, H, HV, 128, V, torch.float32, seed=3)
    clean = _to(inp, dev)
    want = _call(gdn_tree_chunk_update, clean, width)
    request, node = n // 2, 5
    at = request * len(tree) + node
    {"v": inp["v"][0, at, 1], "k": inp["k"][0, at, 0], "a": inp["a"][at]}[what][1] = float("nan")  # column 1, the odd one
    g = _to(inp, dev)
    g["records"].fill_(0.0)
    got = _call(gdn_tree_chunk_update, g, width)
    torch.cuda.synchronize()
    hit = torch.zeros(n, len(tree), HV, V, dtype=torch.bool, device=dev)
    below = [node]
    for j in range(node + 1, len(tree)):
        if tree[j] in below:
            below.append(j)
    cols = {"v": (slice(1, 2), slice(1, 2)), "k": (slice(0, HV // H), slice(0, V)), "a": (slice(1, 2), slice(0, V))}[what]
    hit[request][below, cols[0], cols[1]] = True
    flat = hit.view(n * len(tree), HV, V)
    assert torch.equal(got[0].isnan(), flat)
    assert torch.equal(got[0][~flat], want[0][~flat])
    rows = inp["record_indices"].long()
    assert torch.equal(g["records"][rows, : len(tree), :, :V].isnan(), hit)


@pytest.mark.parametrize("dims,n", [((1, 2, 128, 32), 1), ((2, 16, 64, 64), 16)])  # one and two column tiles a wave
def test_rows_whose_norm_overflows_are_zero_rows(dev, dims, n):
    """Finite keys and queries of magnitude 1e30: their squared norm is infinite in fp32, so they normalise to zero, as in
    the recurrence; nothing becomes NaN."""
    from eagle_harness.kernels.gdn_tree_records import gdn_tree_chunk_update

    announce(f"records chunk form, overflowing norms {dims}")
    tree = [-1, 0, 1, 2, 0, 4, 5] + list(range(6, 30)) + [0, 31, 32]
    got = []
    for big in (True, False):
        inp, width = _inputs([tree] * n, *dims, torch.float32, seed=4)
        for i in range(n):
            for what, node in (("k", 5), ("k", 20), ("q", 3), ("q", 20)):
                row = inp[what][0, i * len(tree) + node]
                row[:] = torch.sign(row) * 1e30 if big else 0.0
        g = _to(inp, dev)
        out = _call(gdn_tree_chunk_update, g, width)
        got.append((out, g["records"]))
    assert not got[0][0].isnan().any()
    assert torch.equal(got[0][0], got[1][0])
    assert torch.equal(got[0][1], got[1][1])


@pytest.mark.parametrize("dims,n", [((1, 2, 128, 32), 1), ((2, 16, 64, 64), 16)])
def test_an_infinite_value_keeps_its_own_delta(dev, dims, n):
    """An infinite value's delta is that infinity; its node's output and everything below in that column are NaN, from
    states that hold infinities of both signs."""
    from eagle_harness.kernels.gdn_tree_records import gdn_tree_chunk_update

    announce(f"records chunk form, infinite value {dims}")
    tree = [-1, 0, 1, 2, 0, 4, 5] + list(range(6, 30)) + [0, 31, 32]
    inp, width = _inputs([tree] * n, *dims, torch.float32, seed=5)
    for i in range(n):
        inp["v"][0, i * len(tree) + 5, 1, 3] = -float("inf")
        inp["v"][0, i * len(tree) + 9, 1, 3] = float("inf")  # below the first
    g = _to(inp, dev)
    out = _call(gdn_tree_chunk_update, g, width)
    below = [5]
    for j in range(6, len(tree)):
        if tree[j] in below:
            below.append(j)
    hit = torch.zeros(len(tree), *out.shape[2:], dtype=torch.bool)
    hit[below, 1, 3] = True
    for i in range(n):
        rec = g["records"][int(inp["record_indices"][i]), : len(tree), :, : dims[3]].cpu()
        assert rec[5, 1, 3] == -float("inf")
        assert torch.equal(rec.isnan(), hit & (torch.arange(len(tree)) != 5)[:, None, None])
        assert torch.equal(out[0, i * len(tree) : (i + 1) * len(tree)].cpu().isnan(), hit)
