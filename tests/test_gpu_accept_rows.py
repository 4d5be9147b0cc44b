"""Greedy targets over rows that start anywhere in a 16-byte line, with ties, infinities and NaN at the edges of the
vectorised part, and the tree walk at the edges of a wave (64 rows) and past it: exact, against the oracle."""

import numpy as np
import pytest
import torch

from conftest import announce
from oracle import accept as oacc
from workloads import seeded_tree

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("vocab", [1, 3, 7, 8, 9, 515, 4097, 102399, 102401])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_targets_of_rows_on_any_boundary(dev, vocab, dtype):
    from eagle_harness.vllm.tree_accept import greedy_targets

    announce(f"argmax vocab={vocab} {dtype}")
    rows = 19
    flat = torch.randn(rows * vocab + 9, generator=torch.Generator().manual_seed(vocab)).to(dtype)
    for shift in (0, 1, 5):
        logits = flat[shift : shift + rows * vocab].clone().view(rows, vocab)
        logits[1] = 0.0  # ties: the first index
        logits[2, -1] = float("inf")
        logits[3] = float("-inf")
        logits[4, vocab // 2] = float("nan")
        logits[5, 0], logits[5, -1] = float("nan"), float("inf")
        logits[6, vocab // 3 :] = 7.0  # a tie across vectors and threads
        held = torch.empty(rows * vocab + 9, dtype=dtype, device=dev)
        held[shift : shift + rows * vocab] = logits.reshape(-1).to(dev)
        got = greedy_targets(held[shift : shift + rows * vocab].view(rows, vocab))
        assert got.tolist() == oacc.argmax_rows(logits).tolist(), shift


@pytest.mark.parametrize("width", [1, 16, 63, 64, 65, 80])
def test_walk_over_trees_of_any_width(dev, width):
    from eagle_harness.vllm.tree_accept import accept_tree
    from eagle_harness.vllm.verify_layout import TreeStore

    announce(f"accept walk width={width}")
    rng = np.random.default_rng(width)
    sizes = [width, 1, 0, max(1, width // 2), width]
    cu = torch.tensor([0] + np.cumsum(sizes).tolist(), dtype=torch.int32)
    n, slots = len(sizes), len(sizes) + 2
    idx = torch.tensor([3, 0, 6, 1, 5], dtype=torch.int32)
    parents = torch.full((slots, width), -1, dtype=torch.int32)
    target = torch.from_numpy(rng.integers(0, 4, sum(sizes)))
    drafted = torch.from_numpy(rng.integers(0, 4, sum(sizes)))
    for b, size in enumerate(sizes):
        if size:
            parents[idx[b], :size] = torch.tensor(seeded_tree(rng, size), dtype=torch.int32)
    last = sizes[0] + sizes[1] + sizes[2] + sizes[3]
    parents[idx[4]] = torch.arange(-1, width - 1, dtype=torch.int32)  # a chain that is accepted to its end
    drafted[last + 1 :] = target[last : last + width - 1]
    store = TreeStore(slots, width, dev)
    sampled, count = accept_tree(target.to(dev), drafted.to(dev), cu.to(dev), idx.to(dev), parents.to(dev), store)
    for b, size in enumerate(sizes):
        path, node = [], 0 if size else None
        while node is not None and len(path) < width:
            path.append(node)
            tok = int(target[int(cu[b]) + node])
            node = next((r for r in range(1, size) if int(parents[idx[b], r]) == node
                         and int(drafted[int(cu[b]) + r]) == tok), None)
        assert int(count[b]) == int(store.path_len[idx[b]]) == len(path)
        assert store.path[idx[b], : len(path)].tolist() == path
        assert sampled[b, : len(path)].tolist() == [int(target[int(cu[b]) + j]) for j in path]
