"""The 16-bit conversions of the kernels' stores against torch's rounding (to nearest even): ties and their neighbours,
subnormals, overflow to infinity, infinities and NaN. Packed (two values to a word) through the records commit, whose fold
of one record with delta 1 into a zero state stores the record's key; one by one through the Mamba2 update's output,
which is D x with C zero and x one."""

import numpy as np
import pytest
import torch

from conftest import announce

pytestmark = pytest.mark.gpu


def _patterns(every):
    """fp32 values: every sign and exponent with leading significands, each with low bits at and around the ties of a
    16-bit result (bf16 drops 16 bits, fp16 13 of a normal value and more of a subnormal one)."""
    high = np.arange(0, 65536, every, dtype=np.uint32) << 16
    low = np.array([0, 1, 0x0FFF, 0x1000, 0x1001, 0x2FFF, 0x3000, 0x3001, 0x7FFF, 0x8000, 0x8001, 0xFFFF], dtype=np.uint32)
    return torch.from_numpy((high[:, None] | low[None]).reshape(-1).view(np.float32).copy())


def _same(got, want):
    assert torch.equal(got.isnan(), want.isnan())
    keep = ~want.isnan()
    assert torch.equal(got[keep], want[keep])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_packed(dev, dtype):
    from eagle_harness.kernels.gdn_tree_records import gdn_tree_records_commit

    announce(f"packed conversion {dtype}")
    K, V, HV = 128, 8, 64
    values = _patterns(1)
    n = values.numel() // (K * HV)
    assert n * K * HV == values.numel()
    records = torch.zeros(1, n, 1, HV, V + K + 1)
    records[..., :V] = 1.0
    records[..., V : V + K] = values.view(1, n, 1, HV, K)
    records[..., V + K] = 1.0
    state = torch.zeros(1, n, HV, V, K, dtype=dtype, device=dev)
    every = torch.arange(n, device=dev)
    gdn_tree_records_commit(state, records.to(dev), every, every, torch.zeros_like(every),
                            torch.full((n, 1), -1, device=dev), True)
    want = values.to(dtype).view(n, HV, 1, K).expand(n, HV, V, K)
    _same(state[0].cpu(), want)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_scalar(dev, dtype):
    from eagle_harness.kernels.mamba2_tree import mamba2_tree_state_update

    announce(f"scalar conversion {dtype}")
    D = _patterns(16)
    heads, hd, ds = D.numel(), 16, 64
    ones = torch.ones(1, heads, hd, dtype=dtype, device=dev)
    state = torch.zeros(2, heads, hd, ds, device=dev)
    out = torch.zeros_like(ones)
    BC = torch.zeros(1, 1, ds, dtype=dtype, device=dev)
    mamba2_tree_state_update(state, ones, torch.zeros(1, heads, dtype=dtype, device=dev), -torch.ones(heads, device=dev),
                             BC, BC, D.to(dev), torch.zeros(heads, device=dev), out,
                             state_indices=torch.ones(1, 1, dtype=torch.int32, device=dev),
                             parents=torch.full((1, 1), -1, dtype=torch.int32, device=dev),
                             query_start_loc=torch.tensor([0, 1], dtype=torch.int32, device=dev))
    _same(out[0].cpu(), D.to(dtype)[:, None].expand(heads, hd))
