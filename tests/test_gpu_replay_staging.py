"""The rounded path replay's staged-node counts (16, 32, 64) and row tiles per wave (one; two for enough heads of V 128),
against the oracle: 16-bit tolerances as the replay's other tests. Requests without records and without a slot among them."""

import numpy as np
import pytest
import torch

from conftest import announce
from oracle import records as orec
from test_gpu_records import _call, _compare, _inputs, _to
from workloads import seeded_tree

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("width,n,dims,dtype", [
    (17, 4, (2, 4, 128, 128), torch.bfloat16), (32, 3, (1, 2, 64, 48), torch.float16), (25, 3, (1, 2, 256, 32), torch.bfloat16),
    (31, 3, (1, 1, 32, 16), torch.bfloat16), (24, 22, (2, 12, 128, 128), torch.bfloat16), (18, 9, (4, 16, 128, 256), torch.float16),
    (33, 3, (1, 2, 128, 64), torch.bfloat16), (16, 4, (2, 4, 128, 128), torch.float16)])
def test_replay_stagings(dev, width, n, dims, dtype):
    from eagle_harness.kernels.gdn_tree_records import gdn_tree_records_update

    announce(f"replay staging width={width} n={n} dims={dims} {dtype}")
    rng = np.random.default_rng(width)
    trees = [seeded_tree(rng, max(1, width - i % 5)) for i in range(n)]
    trees[-1] = list(range(-1, width - 1))
    inp, width = _inputs(trees, *dims, dtype, in_dtype=dtype, seed=width, width=width)
    inp["state_indices"][1] = -1
    inp["record_indices"][0] = -1
    want_rec = inp["records"].clone()
    want = orec.gdn_tree_records_update(inp["A_log"], inp["dt_bias"], inp["q"], inp["k"], inp["v"], inp["a"], inp["b"],
                                        state=inp["state"], state_indices=inp["state_indices"],
                                        query_start_loc=inp["query_start_loc"], parent=inp["parent"],
                                        tree_paths=inp["tree_paths"], records=want_rec,
                                        record_indices=inp["record_indices"], width=width)
    g = _to(inp, dev)
    got = _call(gdn_tree_records_update, g, width, tree_paths=g["tree_paths"])
    torch.cuda.synchronize()
    _compare(got, want, g["records"], want_rec, False, dims[2], dims[3])


@pytest.mark.parametrize("n,dims,dtype", [(3, (2, 4, 128, 128), torch.bfloat16), (22, (2, 12, 128, 128), torch.float16),
                                          (3, (1, 2, 64, 48), torch.bfloat16), (2, (1, 1, 32, 16), torch.bfloat16)])
def test_staged_counts_agree(dev, n, dims, dtype):
    """The same trees under tables of 32 and of 40 columns (32 and 64 staged nodes): the same outputs and records, bit for bit."""
    from eagle_harness.kernels.gdn_tree_records import gdn_tree_records_update

    announce(f"replay staged counts n={n} dims={dims} {dtype}")
    rng = np.random.default_rng(n)
    trees = [seeded_tree(rng, 17 + 5 * i % 16) for i in range(n)]
    got = []
    for width in (32, 40):
        inp, _ = _inputs(trees, *dims, dtype, in_dtype=dtype, seed=n, width=width)
        g = _to(inp, dev)
        out = _call(gdn_tree_records_update, g, width, tree_paths=g["tree_paths"])
        got.append((out, g["records"][:, :32]))
    assert torch.equal(got[0][0], got[1][0])
    assert torch.equal(got[0][1], got[1][1])
