"""The chunk form where its triangular systems are hard: keys alike along the paths, beta near 1 and slow decay, against
the recurrence walked in 64 bits. There the powers of L grow into the thousands, so an inverse formed from them loses
three digits, while the deltas stay of order one and the recurrence itself keeps all of them."""

import numpy as np
import pytest
import torch

from conftest import announce
from test_gpu_records import _call, _inputs, _relabelled_tree, _to
from workloads import seeded_tree

pytestmark = pytest.mark.gpu


def _walk64(inp, width, K, V):
    """Deltas [N, width, HV, V] and outputs [tokens, HV, V] of the recurrence, every node from its parent's state."""
    k, q, v = (inp[x][0].double() for x in "kqv")
    unit = lambda t: t / torch.sqrt((t * t).sum(-1, keepdim=True) + 1e-6)  # noqa: E731
    k, q = unit(k), unit(q) * K**-0.5
    group = v.shape[1] // k.shape[1]
    k, q = k.repeat_interleave(group, 1), q.repeat_interleave(group, 1)
    decay = torch.exp(-torch.exp(inp["A_log"].double()) * torch.nn.functional.softplus(inp["a"].double() + inp["dt_bias"].double()))
    beta = torch.sigmoid(inp["b"].double()).to(inp["b"].dtype).double()  # the gate is of b's type
    delta, out = torch.zeros(*inp["parent"].shape, v.shape[1], V, dtype=torch.float64), torch.zeros_like(v)
    for n, start in enumerate(inp["query_start_loc"][:-1].tolist()):
        size, states = int(inp["query_start_loc"][n + 1]) - start, {}
        first = inp["state"][int(inp["state_indices"][n])].double()
        while len(states) < size:
            for j in range(size):
                p = int(inp["parent"][n, j]) if j else -1
                if j in states or not (p < 0 or p in states):
                    continue
                t = start + j
                h = (first if p < 0 else states[p]) * decay[t, :, None, None]
                delta[n, j] = (v[t] - (h * k[t, :, None]).sum(-1)) * beta[t, :, None]
                states[j] = h + delta[n, j][..., None] * k[t, :, None]
                out[t] = (states[j] * q[t, :, None]).sum(-1)
    return delta, out


@pytest.mark.parametrize("alike,b,a", [(0.9, 8.0, -8.0), (0.99, 4.0, -4.0), (0.999, 8.0, -12.0), (0.5, 8.0, -8.0)])
@pytest.mark.parametrize("width,n,dims,pool_dtype", [
    (40, 3, (1, 2, 128, 32), torch.float32), (64, 2, (2, 2, 64, 16), torch.bfloat16), (24, 2, (1, 2, 32, 48), torch.float16),
    (48, 8, (4, 32, 128, 64), torch.float32),  # two column tiles a wave
    (16, 3, (1, 2, 128, 32), torch.float32), (13, 4, (2, 2, 256, 16), torch.bfloat16),  # one tile of nodes
    (9, 32, (4, 16, 64, 32), torch.float32), (16, 64, (4, 16, 128, 64), torch.bfloat16)])  # two and four column tiles
def test_alike_keys_keep_their_deltas(dev, alike, b, a, width, n, dims, pool_dtype):
    from eagle_harness.kernels.gdn_tree_records import gdn_tree_chunk_update

    announce(f"records chunk form, keys {alike} alike, beta logit {b}, gate {a}, width {width} {dims} {pool_dtype}")
    rng = np.random.default_rng(width)
    trees = [list(range(-1, width - 1)), _relabelled_tree(rng, width)] + [seeded_tree(rng, width - i) for i in range(n - 2)]
    inp, width = _inputs(trees, *dims, pool_dtype, seed=int(1000 * alike))
    gen = torch.Generator().manual_seed(7)
    heads, value_heads, K, V = dims
    inp["k"] = (alike * torch.randn(1, 1, heads, K, generator=gen) + (1 - alike) * inp["k"].float()).bfloat16()
    inp["a"], inp["b"] = torch.full_like(inp["a"], a), torch.full_like(inp["b"], b)
    want, want_out = _walk64(inp, width, K, V)
    g = _to(inp, dev)
    out = _call(gdn_tree_chunk_update, g, width)
    got = g["records"].cpu()[inp["record_indices"].long()][..., :V].double()
    # A delta is a sum over at most 63 ancestors of terms |L| |D|, |L| <= 1 and |D| up to 6 here, each with about five
    # roundings of 2^-24 relative: 63 x 5 x 6 x 6e-8 = 1.1e-4 if all of one sign, sqrt(315) x 6 x 6e-8 = 6.4e-6 if random.
    for i, tree in enumerate(trees):
        torch.testing.assert_close(got[i, : len(tree)], want[i, : len(tree)], atol=2e-5, rtol=2e-5)
    torch.testing.assert_close(out[0].cpu().double(), want_out, atol=1e-2, rtol=1e-2)  # bf16
