"""Performance cases of the draft-tree verify path: what an engine has this package do in a verify round, through the
public entry points, from one short request to the largest served batches.

A case is a dict of plain values with a ``kind``:

- ``attention``: one full-attention layer's tree verify (``verify_attention``) over a paged cache;
- ``front``: one gated-delta-net layer's tree verify as the engine's hook runs it (``TreeVerify.forward_spec_rows``:
  tree conv, then the snapshot walk on views of its output);
- ``chunk`` / ``replay``: one such layer under the records contract, without and with the pool-dtype rounding;
- ``fold``: the records contract's commit of the accepted nodes over all layers of a model;
- ``rows``: a draft step's or a draft extend's attention (``rows_attention``);
- ``mamba2``: one Mamba2 layer's tree state update;
- ``accept``: greedy targets over the vocabulary and the tree walk;
- ``round``: stage, attention, a gated-delta-net layer, accept and the accepted states' commit, in stream order.

Trees follow the rule of ``workloads.py``: a node's parent is drawn from the earlier nodes with fewer than 4 children
and depth below 12. ``ragged`` gives the requests trees of different sizes (half the width and up).
"""

from __future__ import annotations

import math
import sys
from pathlib import Path
from types import SimpleNamespace

import numpy as np
import torch

PACKAGE = str(Path(__file__).resolve().parent.parent / "eagle-4_amd")
if PACKAGE not in sys.path:
    sys.path.insert(0, PACKAGE)

from eagle_harness.kernels.gdn_tree import gdn_tree_ancestors, gdn_tree_paths_buffer  # noqa: E402
from eagle_harness.kernels.gdn_tree_records import (  # noqa: E402
    gdn_tree_chunk_update, gdn_tree_records_commit, gdn_tree_records_update)
from eagle_harness.kernels.mamba2_tree import mamba2_tree_state_update  # noqa: E402
from eagle_harness.kernels.row_attention import RowsLaunch, program_splits, rows_attention, rows_padded, step_splits  # noqa: E402
from eagle_harness.vllm.gdn_tree_verify import GDNSpecRows, LinearStateCommit, TreeVerify  # noqa: E402
from eagle_harness.vllm.tree_accept import accept_tree, greedy_targets  # noqa: E402
from eagle_harness.vllm.verify_attention import verify_attention  # noqa: E402
from eagle_harness.vllm.verify_layout import TreeStore, VerifyStage, set_stage  # noqa: E402

DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32, "fp8": torch.float8_e4m3fn}
BYTES = {"bf16": 2, "f16": 2, "f32": 4, "fp8": 1}
PAD = 4  # record floats past delta, key and decay, as the engine lays them out (V + K + 4 a record)


# ---- the cases -----------------------------------------------------------------------------------------------------
def listed():
    gdn = dict(h=16, hv=32, state="f32")
    return [
        # a single user's request, short context, a small dense model's heads: latency
        dict(name="attention_b1", kind="attention", batch=1, width=16, ragged=False, hq=16, hkv=4, d=128, page=16,
             lmin=512, lmax=512, dtype="bf16", cache="bf16"),
        # the serving batch of the headline workload: long prefixes of very different lengths
        dict(name="attention_b64", kind="attention", batch=64, width=16, ragged=False, hq=24, hkv=4, d=256, page=16,
             lmin=1024, lmax=8192, dtype="bf16", cache="bf16"),
        # the largest served batch, quantized cache, ragged trees
        dict(name="attention_fp8_b512", kind="attention", batch=512, width=16, ragged=True, hq=24, hkv=4, d=256,
             page=16, lmin=512, lmax=4096, dtype="bf16", cache="fp8"),
        # a linear-attention layer of a single user's request
        dict(name="front_b1", kind="front", batch=1, width=16, ragged=False, **gdn),
        # the same layer in the serving batch
        dict(name="front_b64", kind="front", batch=64, width=16, ragged=False, **gdn),
        # records contract, 16-bit pool, the batch the serving engine captures
        dict(name="chunk_b32", kind="chunk", batch=32, width=16, ragged=False, h=16, hv=48, pool="bf16"),
        # records contract with the engine's default fp32 pool and trees wider than 16 nodes, every size different
        dict(name="chunk_wide_b8", kind="chunk", batch=8, width=40, ragged=True, h=16, hv=32, pool="f32"),
        # records contract with the pool's rounding at every node
        dict(name="replay_b32", kind="replay", batch=32, width=16, ragged=True, h=16, hv=48, pool="bf16"),
        # the round's end: accepted nodes of every request folded into the pools of all the model's layers
        dict(name="fold_b16", kind="fold", batch=16, width=16, layers=12, h=16, hv=48, pool="bf16"),
        # a draft step's frontier rows over a sliding window of the committed context
        dict(name="rows_step_b64", kind="rows", batch=64, rows=4, step=7, window=4096, length=8192, hq=32, hkv=8,
             d=128, page=1, dtype="bf16"),
        # a Mamba2 layer's tree verify
        dict(name="mamba2_b16", kind="mamba2", batch=16, width=16, ragged=True, heads=64, hd=64, groups=8, ds=128,
             state="f32"),
        # a whole verify round of one attention and one linear-attention layer at a small serving batch
        dict(name="round_b16", kind="round", batch=16, width=16, ragged=False, hq=24, hkv=4, d=256, page=16,
             lmin=512, lmax=4096, dtype="bf16", cache="bf16", vocab=151936, **gdn),
    ]


def _log(rng, lo, hi):
    """A whole number between ``lo`` and ``hi``, even over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


KINDS = ("attention",) * 4 + ("front",) * 2 + ("chunk",) * 2 + ("rows",) * 2 + ("replay", "fold", "mamba2", "accept", "round")
ATTENTION_HEADS = ((16, 4, 128), (24, 4, 256), (32, 8, 128), (6, 1, 256), (8, 2, 64))
GDN_HEADS = ((16, 32), (16, 48), (4, 8), (4, 12), (2, 6))
MAMBA_HEADS = ((64, 64, 8, 128), (16, 64, 2, 128), (32, 64, 2, 128))


def draw(rng):
    while True:
        kind = rng.choice(KINDS)
        ragged = rng.random() < 0.5
        if kind == "attention":
            hq, hkv, d = rng.choice(ATTENTION_HEADS)
            lmax = _log(rng, 64, 16384)
            dtype, cache = rng.choice((("bf16", "bf16"), ("bf16", "bf16"), ("f16", "f16"), ("bf16", "fp8"), ("f32", "f32")))
            case = dict(kind=kind, batch=_log(rng, 1, 16 if dtype == "f32" else 512), width=rng.randint(3, 32), ragged=ragged,
                        hq=hq, hkv=hkv, d=d, page=rng.choice((16, 16, 64)), lmin=max(16, lmax // rng.choice((1, 2, 8))),
                        lmax=lmax, dtype=dtype, cache=cache)
        elif kind == "front":
            h, hv = rng.choice(GDN_HEADS)
            case = dict(kind=kind, batch=_log(rng, 1, 128), width=rng.randint(3, 32), ragged=ragged, h=h, hv=hv,
                        state=rng.choice(("f32", "f32", "bf16")))
        elif kind == "chunk":
            h, hv = rng.choice(GDN_HEADS)
            case = dict(kind=kind, batch=_log(rng, 1, 128), width=rng.choice((rng.randint(3, 16), rng.randint(17, 64))),
                        ragged=ragged, h=h, hv=hv, pool=rng.choice(("bf16", "f32")))
        elif kind == "replay":
            h, hv = rng.choice(GDN_HEADS)
            case = dict(kind=kind, batch=_log(rng, 1, 64), width=rng.randint(3, 32), ragged=ragged, h=h, hv=hv, pool="bf16")
        elif kind == "fold":
            h, hv = rng.choice(GDN_HEADS)
            case = dict(kind=kind, batch=_log(rng, 1, 64), width=rng.randint(3, 32), layers=_log(rng, 1, 36), h=h, hv=hv,
                        pool=rng.choice(("bf16", "f32")))
        elif kind == "rows":
            hq, hkv, d = rng.choice(((32, 8, 128), (16, 4, 128), (8, 2, 64), (24, 4, 256)))
            step = rng.choice((0, rng.randint(1, 11)))
            case = dict(kind=kind, batch=_log(rng, 1, 96), rows=rng.randint(1, 16 if step == 0 else 8), step=step,
                        window=rng.choice((0, 2048, 4096)), length=_log(rng, 100, 8192), hq=hq, hkv=hkv, d=d,
                        page=rng.choice((1, 16)), dtype=rng.choice(("bf16", "f16")))
        elif kind == "mamba2":
            heads, hd, groups, ds = rng.choice(MAMBA_HEADS)
            case = dict(kind=kind, batch=_log(rng, 1, 64), width=rng.randint(3, 24), ragged=ragged, heads=heads, hd=hd,
                        groups=groups, ds=ds, state=rng.choice(("f32", "bf16")))
        elif kind == "accept":
            case = dict(kind=kind, batch=_log(rng, 1, 128), width=rng.randint(3, 24), ragged=ragged,
                        vocab=rng.choice((32000, 50257, 128256, 151936)), dtype=rng.choice(("bf16", "f32")))
        else:
            hq, hkv, d = rng.choice(ATTENTION_HEADS)
            h, hv = rng.choice(GDN_HEADS)
            lmax = _log(rng, 64, 8192)
            case = dict(kind=kind, batch=_log(rng, 1, 32), width=rng.randint(3, 24), ragged=ragged, hq=hq, hkv=hkv, d=d,
                        page=16, lmin=max(16, lmax // 4), lmax=lmax, dtype="bf16", cache="bf16", vocab=151936, h=h,
                        hv=hv, state="f32")
        w = work(case)
        if w["bytes"] < 1.6e9 and w["flops"] < 1.5e11:
            return case


# ---- what a pass cannot do without ---------------------------------------------------------------------------------
def _mean_rows(case):
    w = case["width"]
    return (math.ceil(w / 2) + w) / 2 if case.get("ragged") else w


def _attention_work(c):
    tokens, ctx = c["batch"] * _mean_rows(c), (c["lmin"] + c["lmax"]) / 2
    e, ec = BYTES[c["dtype"]], BYTES[c["cache"]]
    byte = (c["batch"] * ctx * c["hkv"] * c["d"] * 2 * ec + tokens * (2 * c["hq"] + 2 * c["hkv"]) * c["d"] * e
            + c["batch"] * ctx / c["page"] * 4)
    return byte, 4 * tokens * (ctx + _mean_rows(c) / 2) * c["hq"] * c["d"]


def _front_work(c, k=128, v=128):
    b, tokens, dim = c["batch"], c["batch"] * _mean_rows(c), 2 * c["h"] * k + c["hv"] * v
    state = c["hv"] * k * v * BYTES[c["state"]]
    byte = ((b + tokens) * state + tokens * dim * 2 + b * dim * (3 + c["width"] + 2) * 2 + tokens * c["hv"] * (v + 2) * 2)
    return byte, tokens * (c["hv"] * k * v * 7 + dim * 8)


def _records_work(c, k=128, v=128):
    b, tokens = c["batch"], c["batch"] * _mean_rows(c)
    byte = (b * c["hv"] * k * v * BYTES[c["pool"]] + tokens * (2 * c["h"] * k + 2 * c["hv"] * v + 2 * c["hv"]) * 2
            + tokens * c["hv"] * (v + k + 1) * 4)
    return byte, tokens * c["hv"] * k * v * 7


def _accept_work(c):
    tokens = c["batch"] * _mean_rows(c)
    return tokens * c["vocab"] * BYTES[c["dtype"]] + tokens * 8, tokens * c["vocab"]


def work(case):
    c = case
    if c["kind"] == "attention":
        byte, flops = _attention_work(c)
    elif c["kind"] == "front":
        byte, flops = _front_work(c)
    elif c["kind"] in ("chunk", "replay"):
        byte, flops = _records_work(c)
    elif c["kind"] == "fold":
        depth, n = math.log2(c["width"]) + 1, c["batch"] * c["layers"] * c["hv"]
        byte = n * (2 * 128 * 128 * BYTES[c["pool"]] + depth * 257 * 4)
        flops = n * depth * 128 * 128 * 3
    elif c["kind"] == "rows":
        keys = min(c["length"], c["window"]) if c["window"] > 0 else c["length"]
        own = c["rows"] * c["step"] if c["step"] else c["rows"]
        byte = c["batch"] * ((keys + own) * (c["hkv"] * c["d"] * 2 * 2 + 4) + 2 * c["rows"] * c["hq"] * c["d"] * 2)
        flops = 4 * c["batch"] * c["rows"] * c["hq"] * c["d"] * keys
    elif c["kind"] == "mamba2":
        tokens, state = c["batch"] * _mean_rows(c), c["heads"] * c["hd"] * c["ds"]
        byte = (c["batch"] + tokens) * state * BYTES[c["state"]] + tokens * (2 * c["heads"] * c["hd"] + 2 * c["groups"] * c["ds"] + c["heads"]) * 2
        flops = tokens * state * 5
    elif c["kind"] == "accept":
        byte, flops = _accept_work(c)
    else:
        parts = [_attention_work(c), _front_work(c), _accept_work(c), (c["batch"] * 2 * c["hv"] * 128 * 128 * 4 / 2, 0)]
        byte, flops = (sum(p[i] for p in parts) for i in (0, 1))
    return {"bytes": byte, "flops": flops}


def tolerance(case):
    k = case["kind"]
    if k == "accept":
        return "exact"  # tokens and row numbers
    if k == "attention":
        return {"rel": 2e-5, "max": 2e-3} if case["dtype"] == "f32" else {"rel": 1e-2, "max": 0.1}
    if k == "fold":
        # fp32 sums of the path in another order; a 16-bit pool rounds after every node
        return {"rel": 1e-5, "max": 1e-3} if case["pool"] == "f32" else {"rel": 1e-2, "max": 0.1}
    # 16-bit outputs, and states that follow 16-bit conv outputs or matrix products of 16-bit operands
    return {"rel": 1e-2, "max": 0.1}


# ---- inputs --------------------------------------------------------------------------------------------------------
def _tree(rng, n):
    parents, depth, kids = [-1], [0], [0]
    for _ in range(1, n):
        ok = [j for j in range(len(parents)) if kids[j] < 4 and depth[j] < 12]
        p = ok[int(rng.integers(len(ok)))]
        parents.append(p)
        depth.append(depth[p] + 1)
        kids[p] += 1
        kids.append(0)
    return parents


class _Trees:
    """The batch's trees and their tables on the GPU, in the forms that the engine's stage leaves them in."""

    def __init__(self, case, rng, dev):
        b, w = case["batch"], case["width"]
        # the sizes follow from the case alone, so that every seed has the same number of rows
        own = np.random.default_rng(1000 * b + w)
        sizes = [int(own.integers(math.ceil(w / 2), w + 1)) for _ in range(b)] if case.get("ragged") else [w] * b
        self.lists = [_tree(rng, n) for n in sizes]
        self.sizes, self.width, self.tokens = sizes, w, sum(sizes)
        par = np.full((b, w), -1, np.int32)
        anc = np.full((b, 3, w), -1, np.int32)
        mask = np.zeros((b, w), np.uint64)
        for i, tree in enumerate(self.lists):
            codes = [(-1, -2, -3)]
            for j, p in enumerate(tree):
                par[i, j] = p
                if j:
                    codes.append((p, codes[p][0], codes[p][1]))
                anc[i, :, j] = codes[j]
                mask[i, j] = (1 << j) | (int(mask[i, p]) if p >= 0 else 0)
        start = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int32)
        self.start_list = start.tolist()
        put = lambda x: torch.from_numpy(x).to(dev)  # noqa: E731
        self.parents, self.ancestors, self.masks, self.start = put(par), put(anc), put(mask.view(np.int64)), put(start)


def _generator(seed, dev):
    return torch.Generator(device=dev).manual_seed(seed)


def _attention_state(c, rng, gen, dev, trees):
    b, dt = c["batch"], DTYPES[c["dtype"]]
    lens = rng.integers(c["lmin"], c["lmax"] + 1, b)
    pages = [-(-int(n) // c["page"]) for n in lens]
    total = sum(pages) + 1
    order = rng.permutation(total).astype(np.int32)
    table, at = np.full((b, max(pages)), order[-1], np.int32), 0
    for i, n in enumerate(pages):
        table[i, :n] = order[at : at + n]
        at += n
    randn = lambda *s: torch.randn(*s, device=dev, generator=gen)  # noqa: E731
    x = dict(q=(randn(trees.tokens, c["hq"], c["d"]) * 0.5).to(dt), k=(randn(trees.tokens, c["hkv"], c["d"]) * 0.5).to(dt),
             v=(randn(trees.tokens, c["hkv"], c["d"]) * 0.5).to(dt), scales={}, lens=torch.tensor(lens, dtype=torch.int32, device=dev),
             table=torch.from_numpy(table).to(dev), len_list=lens.tolist())
    for name in ("k", "v"):
        cache = randn(total, c["page"], c["hkv"], c["d"])
        if c["cache"] == "fp8":  # one scale per (page, KV head): its largest value is 448
            scale = cache.abs().amax(dim=(1, 3)) / 448.0
            x[name + "_cache"] = (cache / scale[:, None, :, None]).clamp_(-448, 448).to(torch.float8_e4m3fn)
            x["scales"][name + "_scale"] = scale
        else:
            x[name + "_cache"] = cache.mul_(0.5).to(dt)
        del cache
    x["out"] = torch.empty_like(x["q"])
    return x


def _gates(c, tokens, gen, dev):
    """The layer's decay parameters (A in [1, 16], as trained models start) and a / b of every token."""
    hv = c["hv"]
    return dict(A_log=torch.log(1 + 15 * torch.rand(hv, device=dev, generator=gen)),
                dt_bias=torch.randn(hv, device=dev, generator=gen) - 4,
                a=torch.randn(tokens, hv, device=dev, generator=gen).bfloat16(),
                b=torch.randn(tokens, hv, device=dev, generator=gen).bfloat16())


def _front_state(c, rng, gen, dev, trees, k=128, v=128):
    """A layer's input projection [qkv | z | b | a] and its caches: one state slot per verify row, scattered over the
    pool (slot 0 is the engine's null block), the conv window in the slot of row 0."""
    b, w, h, hv = c["batch"], c["width"], c["h"], c["hv"]
    dim = 2 * h * k + hv * v
    g = _gates(c, trees.tokens, gen, dev)
    proj = torch.randn(trees.tokens, dim + hv * v + 2 * hv, device=dev, generator=gen).bfloat16()
    proj[:, dim + hv * v : dim + hv * v + hv] = g["b"]
    proj[:, dim + hv * v + hv :] = g["a"]
    slots = torch.from_numpy(1 + rng.permutation(b * w).astype(np.int32)).view(b, w).to(dev)
    accepted = torch.from_numpy(rng.integers(1, min(w, 5) + 1, b).astype(np.int32)).to(dev)
    pool = torch.zeros(1 + b * w, hv, v, k, dtype=DTYPES[c["state"]], device=dev)
    first = slots.gather(1, accepted.long()[:, None] - 1)[:, 0].long()
    pool[first] = (torch.randn(b, hv, v, k, device=dev, generator=gen) * 0.02).to(pool.dtype)
    conv = torch.zeros(1 + b * w, dim, w + 2, dtype=torch.bfloat16, device=dev)
    conv[slots[:, 0].long()] = torch.randn(b, dim, w + 2, device=dev, generator=gen).bfloat16()
    weight = (torch.randn(dim, 4, device=dev, generator=gen) * 0.3).bfloat16()
    return GDNSpecRows("layers.0.linear_attn", proj[:, :dim], conv, weight, None, "silu", proj[:, dim + hv * v + hv :],
                       proj[:, dim + hv * v : dim + hv * v + hv], g["A_log"], g["dt_bias"], pool, slots, trees.start,
                       accepted, torch.zeros(trees.tokens, hv * v, dtype=torch.bfloat16, device=dev), h, k, hv, v)


def _records_state(c, rng, gen, dev, trees, k=128, v=128):
    b, h, hv = c["batch"], c["h"], c["hv"]
    randn = lambda *s: torch.randn(*s, device=dev, generator=gen)  # noqa: E731
    return dict(_gates(c, trees.tokens, gen, dev), q=randn(1, trees.tokens, h, k).bfloat16(),
                k=randn(1, trees.tokens, h, k).bfloat16(), v=randn(1, trees.tokens, hv, v).bfloat16(),
                state=(randn(b + 1, hv, v, k) * 0.02).to(DTYPES[c["pool"]]),
                slots=torch.from_numpy(1 + rng.permutation(b).astype(np.int32)).to(dev),
                records=torch.zeros(b, c["width"], hv, v + k + PAD, device=dev),
                rows=torch.from_numpy(rng.permutation(b).astype(np.int32)).to(dev))


def _path_table(x, c, trees, dev):
    """The replay's path table, as the engine derives it from its first-child / next-sibling links."""
    b, w = c["batch"], c["width"]
    first, sibling = np.full((b, w), -1, np.int64), np.full((b, w), -1, np.int64)
    for i, tree in enumerate(trees.lists):
        last = {}
        for j, p in enumerate(tree):
            if j == 0:
                continue
            if p in last:
                sibling[i, last[p]] = j
            else:
                first[i, p] = j
            last[p] = j
    paths = gdn_tree_paths_buffer(b, w, dev)
    gdn_tree_ancestors(torch.from_numpy(first).to(dev), torch.from_numpy(sibling).to(dev), trees.parents.long(), x["slots"], w,
                       torch.empty(b, 3, w, dtype=torch.int32, device=dev), trees.start, paths)
    return paths


def _logits_state(c, rng, gen, dev, trees):
    """Logits with a clear winner in every row, and drafts that agree with their parent's at most of the nodes."""
    vocab, dt = c["vocab"], DTYPES[c["dtype"]]
    logits = torch.randn(trees.tokens, vocab, device=dev, generator=gen).to(dt)
    target = rng.integers(0, vocab, trees.tokens)
    logits[torch.arange(trees.tokens, device=dev), torch.from_numpy(target).to(dev)] = 20.0
    drafted = rng.integers(0, vocab, trees.tokens)
    for s, tree in zip(trees.start_list, trees.lists):
        for j, p in enumerate(tree):
            if j and rng.random() < 0.7:
                drafted[s + j] = target[s + p]
    paths = []
    for s, tree in zip(trees.start_list, trees.lists):
        path = [0]
        while True:
            kid = next((j for j, p in enumerate(tree) if j and p == path[-1] and drafted[s + j] == target[s + path[-1]]), None)
            if kid is None:
                break
            path.append(kid)
        paths.append(path)
    return dict(logits=logits, drafted=torch.from_numpy(drafted).to(dev), paths=paths)


def prepare(case, seed):
    c = case
    dev = torch.device("cuda", torch.cuda.current_device())
    rng, gen = np.random.default_rng(seed), _generator(seed, dev)
    s = SimpleNamespace(case=c, dev=dev)
    if c["kind"] == "rows":
        _rows_state(s, c, rng, gen, dev)
        return s
    s.trees = _Trees(c, rng, dev)
    if c["kind"] in ("attention", "round"):
        s.att = _attention_state(c, rng, gen, dev, s.trees)
    if c["kind"] in ("front", "round"):
        s.rows = _front_state(c, rng, gen, dev, s.trees)
        s.layer = TreeVerify()
        s.stage = SimpleNamespace(ancestors=s.trees.ancestors, parents=s.trees.parents, state_slots={})
    if c["kind"] in ("accept", "round"):
        s.heads = _logits_state(c, rng, gen, dev, s.trees)
        s.store = TreeStore(c["batch"], c["width"], dev)
        s.idx = torch.from_numpy(rng.permutation(c["batch"]).astype(np.int32)).to(dev)
        s.store.parents[s.idx.long()] = s.trees.parents
    if c["kind"] == "round":

        s.stage = VerifyStage(c["batch"], s.trees.tokens, c["width"], dev)
        s.positions = torch.cat([torch.arange(n, device=dev) + int(l) for n, l in zip(s.trees.sizes, s.att["len_list"])])
        s.commit = LinearStateCommit([(s.rows.conv_state, s.rows.ssm_state)], [s.rows.state_indices], dev)
    if c["kind"] in ("chunk", "replay"):
        s.x = _records_state(c, rng, gen, dev, s.trees)
        if c["kind"] == "replay":
            s.paths = _path_table(s.x, c, s.trees, dev)
    if c["kind"] == "fold":
        b, hv, L = c["batch"], c["hv"], c["layers"]
        s.state = torch.empty(L, b + 1, hv, 128, 128, dtype=DTYPES[c["pool"]], device=dev)
        s.records = torch.zeros(L, b, c["width"], hv, 256 + PAD, device=dev)
        for i in range(L):
            s.state[i] = (torch.randn(b + 1, hv, 128, 128, device=dev, generator=gen) * 0.02).to(s.state.dtype)
            s.records[i, ..., :128] = torch.randn(b, c["width"], hv, 128, device=dev, generator=gen) * 0.5
            key = torch.randn(b, c["width"], hv, 128, device=dev, generator=gen)
            s.records[i, ..., 128:256] = key / key.norm(dim=-1, keepdim=True)
            s.records[i, ..., 256] = torch.rand(b, c["width"], hv, device=dev, generator=gen) * 0.2 + 0.8
        s.slots = torch.from_numpy(1 + rng.permutation(b).astype(np.int32)).to(dev)
        s.rec_rows = torch.from_numpy(rng.permutation(b).astype(np.int32)).to(dev)
        s.node = torch.from_numpy(rng.integers(0, c["width"], b).astype(np.int32)).to(dev)
    if c["kind"] == "mamba2":
        b, w, t, H, P, G, N = c["batch"], c["width"], s.trees.tokens, c["heads"], c["hd"], c["groups"], c["ds"]
        randn = lambda *z: torch.randn(*z, device=dev, generator=gen)  # noqa: E731
        s.slots = torch.from_numpy(1 + rng.permutation(b * w).astype(np.int32)).view(b, w).to(dev)
        s.accepted = torch.from_numpy(rng.integers(1, min(w, 5) + 1, b).astype(np.int32)).to(dev)
        s.state = torch.zeros(1 + b * w, H, P, N, dtype=DTYPES[c["state"]], device=dev)
        s.state[s.slots.gather(1, s.accepted.long()[:, None] - 1)[:, 0].long()] = (randn(b, H, P, N) * 0.1).to(s.state.dtype)
        s.mixed = randn(t, H * P + 2 * G * N).bfloat16()  # the conv's output: x, B and C are views of it
        s.dt = randn(t, H).bfloat16()
        s.A, s.D, s.bias = -(1 + 15 * torch.rand(H, device=dev, generator=gen)), randn(H), randn(H) - 3
        s.out = torch.zeros(t, H, P, dtype=torch.bfloat16, device=dev)
    return s


def _rows_state(s, c, rng, gen, dev):
    b, r, step, page, dt = c["batch"], c["rows"], c["step"], c["page"], DTYPES[c["dtype"]]
    own = r * step if step else r
    pages = -(-(c["length"] + own) // page)
    s.lens = rng.integers(max(1, c["length"] // 2), c["length"] + 1, b)
    table = rng.permutation(b * pages).astype(np.int32).reshape(b, pages)
    shape = (b * pages * page, c["hkv"], c["d"]) if page == 1 else (b * pages, page, c["hkv"], c["d"])
    s.keys = torch.randn(*shape, device=dev, generator=gen).to(dt)
    s.values = torch.randn(*shape, device=dev, generator=gen).to(dt)
    s.q = torch.randn(b * r, c["hq"], c["d"], device=dev, generator=gen).to(dt)
    s.out = torch.zeros_like(s.q)
    s.table, s.seq = torch.from_numpy(table).to(dev), torch.tensor(s.lens, dtype=torch.int32, device=dev)
    s.anc = None
    if step:  # the nodes drafted so far take the slots after the committed keys
        at = s.lens[:, None, None] + rng.integers(0, own, (b, r, step))
        s.anc = torch.from_numpy((table[np.arange(b)[:, None, None], at // page] * page + at % page).astype(np.int32)).to(dev)
    splits = step_splits(b * c["hq"], dev) if step else program_splits(b * c["hq"], dev)
    s.launch = RowsLaunch(splits=max(splits, 8), block_n=32)
    parts = b * c["hq"] * (s.launch.splits + 1) * rows_padded(r)
    s.part_out, s.part_lse = torch.empty(parts, c["d"], device=dev), torch.empty(parts, device=dev)


# ---- one pass ------------------------------------------------------------------------------------------------------
def _attend(s, lens, masks):
    x = s.att
    return verify_attention(x["q"], x["k"], x["v"], x["k_cache"], x["v_cache"], x["table"], lens, s.trees.start, masks,
                            s.case["d"] ** -0.5, x["out"], max_query_len=s.case["width"], **x["scales"])


def _layer(s):
    set_stage(s.stage)
    s.layer.forward_spec_rows(s.rows)


def run(s):
    c = s.case
    if c["kind"] == "attention":
        return _attend(s, s.att["lens"], s.trees.masks)
    if c["kind"] == "front":
        _layer(s)
        return {"out": s.rows.out, "states": s.rows.ssm_state, "conv": s.rows.conv_state}
    if c["kind"] in ("chunk", "replay"):
        x = s.x
        args = (x["A_log"], x["dt_bias"], x["q"], x["k"], x["v"], x["a"], x["b"])
        kw = dict(state=x["state"], state_indices=x["slots"], query_start_loc=s.trees.start, parent=s.trees.parents,
                  records=x["records"], record_indices=x["rows"], width=c["width"])
        out = gdn_tree_chunk_update(*args, **kw) if c["kind"] == "chunk" else gdn_tree_records_update(*args, tree_paths=s.paths, **kw)
        return {"out": out, "records": x["records"]}
    if c["kind"] == "fold":
        gdn_tree_records_commit(s.state, s.records, s.slots, s.rec_rows, s.node, s.trees.parents, c["pool"] != "f32")
        return s.state
    if c["kind"] == "rows":
        rows_attention(s.q, s.keys, s.values, s.out, s.part_out, s.part_lse, s.table, s.seq, s.anc,
                       rows_per_request=c["rows"], step=c["step"], window=c["window"], scale=c["d"] ** -0.5,
                       launch=s.launch, table_page=c["page"])
        return s.out
    if c["kind"] == "mamba2":
        H, P, G, N = c["heads"], c["hd"], c["groups"], c["ds"]
        t = s.mixed.shape[0]
        x, B, C = (s.mixed[:, : H * P].view(t, H, P), s.mixed[:, H * P : H * P + G * N].view(t, G, N),
                   s.mixed[:, H * P + G * N :].view(t, G, N))
        mamba2_tree_state_update(s.state, x, s.dt, s.A, B, C, s.D, s.bias, s.out, state_indices=s.slots,
                                 parents=s.trees.parents, query_start_loc=s.trees.start, num_accepted_tokens=s.accepted,
                                 pad_slot_id=0)
        return {"out": s.out, "states": s.state}

    if c["kind"] == "accept":
        target = greedy_targets(s.heads["logits"])
        _, count = accept_tree(target, s.heads["drafted"], s.trees.start, s.idx, s.store.parents, s.store)
        return {"target": target, "count": count, "path": s.store.path, "path_len": s.store.path_len}
    t = s.trees
    s.stage.stage(s.store, s.idx, t.start, t.start, s.positions, c["batch"], t.tokens, tree=True)
    att = _attend(s, s.stage.context_lens[: c["batch"]], s.stage.masks[: c["batch"]])
    _layer(s)
    target = greedy_targets(s.heads["logits"])
    _, count = accept_tree(target, s.heads["drafted"], t.start, s.idx, s.store.parents, s.store)
    s.commit.commit(s.idx, s.store.path, s.store.path_len)
    return {"attention": att, "out": s.rows.out, "states": s.rows.ssm_state, "conv": s.rows.conv_state, "target": target,
            "count": count, "path": s.store.path, "path_len": s.store.path_len, "positions": s.positions}


# ---- the same in 64 bits -------------------------------------------------------------------------------------------
def _attend64(s):
    x, c = s.att, s.case
    page, g = c["page"], c["hq"] // c["hkv"]
    out = torch.zeros(x["q"].shape, dtype=torch.float64, device=s.dev)
    for i, n in enumerate(s.trees.sizes):
        at, l = s.trees.start_list[i], int(x["len_list"][i])
        blocks = x["table"][i, : -(-l // page)].long()

        def rows(name):
            old = x[name + "_cache"][blocks].double()
            if x["scales"]:
                old = old * x["scales"][name + "_scale"][blocks].double()[:, None, :, None]
            return torch.cat([old.flatten(0, 1)[:l], x[name][at : at + n].double()]).permute(1, 0, 2).contiguous()  # [hkv, keys, d]

        keys, values = rows("k"), rows("v")
        q = x["q"][at : at + n].double().view(n, c["hkv"], g, -1).permute(1, 0, 2, 3).reshape(c["hkv"], n * g, -1)
        see = torch.ones(n, l + n, dtype=torch.bool, device=s.dev)
        see[:, l:] = (s.trees.masks[i, :n, None] >> torch.arange(n, device=s.dev)) & 1 == 1
        score = q @ keys.transpose(1, 2).contiguous() * c["d"] ** -0.5
        score.masked_fill_(~see.repeat_interleave(g, 0), -math.inf)
        o = score.softmax(-1) @ values
        out[at : at + n] = o.view(c["hkv"], n, g, -1).permute(1, 0, 2, 3).reshape(n, c["hq"], -1)
    return out


def _padded(s, flat):
    """[tokens, ...] rows as [batch, width, ...] in 64 bits, zeros after each request's last."""
    t = s.trees
    out = torch.zeros(len(t.sizes), t.width, *flat.shape[1:], dtype=torch.float64, device=s.dev)
    for i, n in enumerate(t.sizes):
        out[i, :n] = flat[t.start_list[i] : t.start_list[i] + n].double()
    return out


def _flat(s, padded):
    return torch.cat([padded[i, :n] for i, n in enumerate(s.trees.sizes)])


def _delta64(s, q, k, v, a, b, A_log, dt_bias, first):
    """The gated delta rule over the trees: q, k [tokens, H, K], v [tokens, HV, V], states [batch, width, HV, V, K]."""
    group = v.shape[1] // q.shape[1]
    unit = lambda t: t / torch.sqrt((t * t).sum(-1, keepdim=True) + 1e-6)  # noqa: E731
    q, k, v = unit(_padded(s, q)) * q.shape[-1] ** -0.5, unit(_padded(s, k)), _padded(s, v)
    q, k = q.repeat_interleave(group, 2), k.repeat_interleave(group, 2)
    decay = torch.exp(-torch.exp(A_log.double()) * torch.nn.functional.softplus(_padded(s, a) + dt_bias.double()))
    beta = torch.sigmoid(_padded(s, b)).to(torch.bfloat16).double()  # the gate is of b's type
    batch, width = s.trees.parents.shape
    states = torch.zeros(batch, width, *first.shape[1:], dtype=torch.float64, device=s.dev)
    out, delta, every = torch.zeros_like(v), torch.zeros_like(v), torch.arange(batch, device=s.dev)
    for j in range(width):
        h = first if j == 0 else states[every, s.trees.parents[:, j].long().clamp(min=0)]
        h = h * decay[:, j, :, None, None]
        d = (v[:, j] - (h * k[:, j, :, None, :]).sum(-1)) * beta[:, j, :, None]
        h = h + d[..., None] * k[:, j, :, None, :]
        states[:, j], delta[:, j], out[:, j] = h, d, (h * q[:, j, :, None, :]).sum(-1)
    return out, states, delta, k, decay


def _front64(s):
    r, t = s.rows, s.trees
    k, v, h, hv = r.head_k_dim, r.head_v_dim, r.num_k_heads, r.num_v_heads
    x, w = _padded(s, r.mixed_qkv), r.conv_weight.double()
    every, acc = torch.arange(len(t.sizes), device=s.dev), r.num_accepted_tokens.long()
    window = r.conv_state[r.state_indices[:, 0].long()].double()
    past = torch.stack([window[every, :, acc - 1 + i] for i in range(3)], 1)  # [batch, 3, dim], oldest first
    line = torch.cat([past, x], 1)
    y = x * w[:, 3]
    for i in range(3):
        code = t.ancestors[:, i].long()
        y = y + torch.gather(line, 1, (code + 3)[:, :, None].expand(-1, -1, line.shape[2])) * w[:, 2 - i]
    y = _flat(s, y * torch.sigmoid(y))
    n = y.shape[0]
    pool = r.ssm_state.double()
    first = pool[r.state_indices[every, acc - 1].long()]
    out, states, *_ = _delta64(s, y[:, : h * k].view(n, h, k), y[:, h * k : 2 * h * k].view(n, h, k), y[:, 2 * h * k :].view(n, hv, v),
                               r.a, r.b, r.A_log, r.dt_bias, first)
    for i, m in enumerate(t.sizes):
        pool[r.state_indices[i, :m].long()] = states[i, :m]
    return _flat(s, out).view(n, hv * v), pool


def exact(case, seed):
    c = case
    if c["kind"] == "accept":
        return None
    s = prepare(case, seed)
    if c["kind"] == "attention":
        return _attend64(s)
    if c["kind"] == "front":
        out, pool = _front64(s)
        return {"out": out, "states": pool, "conv": None}
    if c["kind"] in ("chunk", "replay"):
        x = s.x
        out, _, delta, key, decay = _delta64(s, x["q"][0], x["k"][0], x["v"][0], x["a"], x["b"], x["A_log"], x["dt_bias"],
                                             x["state"][x["slots"].long()].double())
        rec = torch.zeros(x["records"].shape, dtype=torch.float64, device=s.dev)
        for i, n in enumerate(s.trees.sizes):
            at = int(x["rows"][i])
            rec[at, :n, :, :128], rec[at, :n, :, 128:256], rec[at, :n, :, 256] = delta[i, :n], key[i, :n], decay[i, :n]
        return {"out": _flat(s, out)[None], "records": rec}
    if c["kind"] == "fold":
        state, node = s.state.double(), s.node.tolist()
        for i, tree in enumerate(s.trees.lists):
            path, at, row = [], int(s.slots[i]), int(s.rec_rows[i])
            j = node[i]
            while j >= 0:
                path.append(j)
                j = tree[j]
            h = state[:, at]
            for j in reversed(path):
                r = s.records[:, row, j].double()
                h = h * r[..., 256, None, None] + r[..., :128, None] * r[..., None, 128:256]
            state[:, at] = h
        return state
    if c["kind"] == "rows":
        g, page, r = c["hq"] // c["hkv"], c["page"], c["rows"]
        out = torch.zeros(s.q.shape, dtype=torch.float64, device=s.dev)
        keys, values = s.keys.view(-1, c["hkv"], c["d"]), s.values.view(-1, c["hkv"], c["d"])
        for i, l in enumerate(s.lens.tolist()):
            for j in range(r):
                last = l - 1 if c["step"] else l + j
                low = max(0, last - c["window"] + 1) if c["window"] > 0 else 0
                at = torch.arange(low, last + 1, device=s.dev)
                at = s.table[i, at // page].long() * page + at % page
                if c["step"]:
                    at = torch.cat([at, s.anc[i, j].long()])
                q = s.q[i * r + j].double().view(c["hkv"], g, -1)
                kk, vv = (z[at].double().permute(1, 0, 2).contiguous() for z in (keys, values))
                out[i * r + j] = ((q @ kk.transpose(1, 2).contiguous() * c["d"] ** -0.5).softmax(-1) @ vv).reshape(c["hq"], -1)
        return out
    if c["kind"] == "mamba2":
        H, P, G, N = c["heads"], c["hd"], c["groups"], c["ds"]
        m = _padded(s, s.mixed)
        b, w = m.shape[:2]
        x = m[..., : H * P].reshape(b, w, H, P)
        B, C = (m[..., H * P + i * G * N : H * P + (i + 1) * G * N].reshape(b, w, G, N).repeat_interleave(H // G, 2) for i in (0, 1))
        dt = torch.nn.functional.softplus(_padded(s, s.dt) + s.bias.double())
        pool, every = s.state.double(), torch.arange(b, device=s.dev)
        first = pool[s.slots[every, s.accepted.long() - 1].long()]
        states, out = torch.zeros(b, w, H, P, N, dtype=torch.float64, device=s.dev), torch.zeros_like(x)
        for j in range(w):
            h = first if j == 0 else states[every, s.trees.parents[:, j].long().clamp(min=0)]
            h = h * torch.exp(s.A.double() * dt[:, j])[..., None, None] + x[:, j, ..., None] * (B[:, j] * dt[:, j, :, None])[:, :, None, :]
            states[:, j], out[:, j] = h, (h * C[:, j, :, None, :]).sum(-1) + x[:, j] * s.D.double()[:, None]
        for i, n in enumerate(s.trees.sizes):
            pool[s.slots[i, :n].long()] = states[i, :n]
        return {"out": _flat(s, out), "states": pool}
    out, pool = _front64(s)
    for i, path in enumerate(s.heads["paths"]):
        last, n = path[-1], len(path)
        if last != n - 1:
            pool[int(s.rows.state_indices[i, n - 1])] = pool[int(s.rows.state_indices[i, last])]
    return {"attention": _attend64(s), "out": out, "states": pool, "conv": None, "target": None, "count": None, "path": None,
            "path_len": None, "positions": None}
