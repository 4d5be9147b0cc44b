"""The merges of split attention at one, four and more runs per row (a few partials to over a hundred), every head dim and
schedule, against the oracle: 16-bit rows 2e-2 abs / 1e-2 rel, fp32 rows 1e-4, as the schedules' other tests."""

import pytest
import torch

from conftest import announce
from oracle import attention as oatt
from oracle import row_attention as orow
from workloads import AttnShape, attention_inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch,lmin,lmax,d,dtype", [
    (1, 700, 700, 128, torch.bfloat16), (1, 1500, 1500, 64, torch.float16), (1, 4090, 4090, 128, torch.bfloat16),
    (1, 4090, 4090, 256, torch.bfloat16), (1, 4000, 4000, 32, torch.bfloat16), (1, 9001, 9001, 64, torch.bfloat16),
    (2, 100, 6000, 128, torch.float16), (3, 20, 5000, 256, torch.bfloat16), (1, 9001, 9001, 32, torch.float16),
    (1, 5000, 5000, 128, torch.float32), (2, 300, 2500, 64, torch.float32), (1, 900, 900, 256, torch.float32)])
def test_verify_attention_over_many_partials(dev, batch, lmin, lmax, d, dtype):
    from eagle_harness.vllm.verify_attention import verify_attention

    announce(f"merge runs batch={batch} L={lmin}..{lmax} D={d} {dtype}")
    x = attention_inputs(AttnShape(batch, 7, 6, 2, d, 16, lmin, lmax), seed=d + batch, dtype=dtype)
    args = lambda t, out: (t["q"], t["k_new"], t["v_new"], t["key_cache"], t["value_cache"], t["block_table"],  # noqa: E731
                           t["context_lens"], t["query_start_loc"], t["masks"], t["scale"], out)
    want = oatt.verify_attention(*args(x, torch.zeros_like(x["q"])), max_query_len=7)
    g = {k: (v.to(dev) if isinstance(v, torch.Tensor) else v) for k, v in x.items()}
    got = verify_attention(*args(g, torch.zeros_like(g["q"])), max_query_len=7)
    tol = dict(atol=1e-4, rtol=1e-4) if dtype == torch.float32 else dict(atol=2e-2, rtol=1e-2)
    torch.testing.assert_close(got.cpu().float(), want.float(), **tol)


@pytest.mark.parametrize("splits,d,step", [(1, 64, 3), (8, 128, 0), (9, 64, 2), (33, 256, 1), (64, 128, 5), (128, 64, 4)])
def test_draft_rows_over_many_splits(dev, splits, d, step):
    from eagle_harness.kernels.row_attention import RowsLaunch, rows_attention, rows_padded

    announce(f"merge runs rows splits={splits} D={d} step={step}")
    gen = torch.Generator().manual_seed(splits)
    bs, rows, heads, kv, length = 2, 3, 4, 2, 700
    slots = bs * (length + 64)
    keys, values = (torch.randn(slots, kv, d, generator=gen).bfloat16() for _ in range(2))
    q = torch.randn(bs * rows, heads, d, generator=gen).bfloat16()
    table = torch.randperm(slots, generator=gen).to(torch.int32).view(bs, -1)
    seq = torch.tensor([length, 33], dtype=torch.int32)  # the second: most splits hold no key
    anc = torch.stack([table[b, int(seq[b]) : int(seq[b]) + rows * max(step, 1)].view(rows, -1) for b in range(bs)]).contiguous()
    kw = dict(rows_per_request=rows, step=step, window=0, scale=d**-0.5)
    want = orow.rows_attention(q, keys, values, table, seq, anc if step else None, **kw)
    parts = bs * heads * (splits + 1) * rows_padded(rows)
    out = torch.empty_like(q, device=dev)
    rows_attention(q.to(dev), keys.to(dev), values.to(dev), out, torch.empty(parts, d, device=dev),
                   torch.empty(parts, device=dev), table.to(dev), seq.to(dev), anc.to(dev) if step else None,
                   launch=RowsLaunch(splits=splits, block_n=32), **kw)
    torch.testing.assert_close(out.cpu().float(), want.float(), atol=2e-2, rtol=1e-2)
