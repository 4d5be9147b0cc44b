"""Verify attention of small jobs, one request (whose short tables take the split schedule) to a few: ragged contexts (empty
ones among them) against the oracle, and several requests under wider block tables, whose results keep their bits. 2e-2
abs / 1e-2 rel, as the schedules' other tests."""

import pytest
import torch

from conftest import announce
from oracle import attention as oatt
from workloads import AttnShape, attention_inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch,lmax,hq,hkv,d,page,fp8", [
    (2, 1000, 8, 2, 64, 16, False), (8, 500, 8, 2, 128, 16, False), (5, 130, 6, 1, 256, 48, False), (3, 95, 4, 1, 32, 7, False),
    (16, 700, 16, 4, 128, 16, False), (9, 2600, 8, 2, 128, 64, False), (3, 900, 24, 4, 256, 16, False),
    (1, 40, 4, 2, 64, 16, True), (2, 1000, 6, 2, 128, 16, True), (12, 600, 6, 1, 256, 64, True), (1, 9000, 4, 2, 64, 16, True)])
def test_small_jobs(dev, batch, lmax, hq, hkv, d, page, fp8):
    from eagle_harness.vllm.verify_attention import verify_attention

    announce(f"attention job batch={batch} L<={lmax} {hq}/{hkv} D={d} page={page} fp8={fp8}")
    x = attention_inputs(AttnShape(batch, 9, hq, hkv, d, page, lmax // 3, lmax), seed=batch + d, fp8=fp8)
    if batch > 2:
        x["context_lens"][1] = 0
    scales = {k: x[k] for k in ("k_scale", "v_scale") if k in x}
    run = lambda fn, t, out, **kw: fn(t["q"], t["k_new"], t["v_new"], t["key_cache"], t["value_cache"], t["block_table"],  # noqa: E731
                                      t["context_lens"], t["query_start_loc"], t["masks"], t["scale"], out,
                                      max_query_len=9, **kw)
    want = run(oatt.verify_attention, x, torch.zeros_like(x["q"]), **scales)
    g = {k: (v.to(dev) if isinstance(v, torch.Tensor) else v) for k, v in x.items()}
    on_dev = {k: g[k] for k in scales}
    got = run(verify_attention, g, torch.zeros_like(g["q"]), **on_dev)
    torch.testing.assert_close(got.cpu().float(), want.float(), atol=2e-2, rtol=1e-2)
    no_alloc = run(verify_attention, g, torch.zeros_like(g["q"]), no_alloc=True, **on_dev)
    assert torch.equal(no_alloc, got)
    if batch > 1:  # the table an engine hands over is as wide as its longest allowed context: nothing follows from its width
        table = g["block_table"]
        g["block_table"] = torch.cat([table, table[:, :1].expand(-1, 3 * table.shape[1] + 5)], 1)
        assert torch.equal(run(verify_attention, g, torch.zeros_like(g["q"]), **on_dev), got)
