"""The work a user of this framework has it do, as cases that can be timed.

Every case goes through the tensor-level entry points (``ops``) the four plugins drive, or, for the prefetch round,
through ``GSAPrefetchEngineC``: representatives of a prompt's blocks, a decode step's retrieval (one layer at a time
as an attention hook makes it, or all layers at once), the gather of what was selected, whole-block dumps and loads,
hash codes, KVStar votes, ESA slot lists, and the prefetch engine's round.  Keys, values and queries are N(0, 1) like
the rest of the repository's inputs; consecutive decode queries of one state drift with correlation 0.95.  The
segment lengths of a case are part of its shape (the same for every seed); block tables, lists and values come from
the seed.
"""
from __future__ import annotations

import importlib.util
import math
import os
import sys

import numpy as np
import torch

PACKAGE, MODULE = "unified-cache-management_amd", "ucm_amd"


def _package():
    """The package's directory is not a python identifier: it is imported under the name ``ucm_amd``."""
    if MODULE not in sys.modules:
        where = os.path.join(os.getcwd(), PACKAGE)
        spec = importlib.util.spec_from_file_location(MODULE, os.path.join(where, "__init__.py"),
                                                      submodule_search_locations=[where])
        mod = importlib.util.module_from_spec(spec)
        sys.modules[MODULE] = mod
        spec.loader.exec_module(mod)
    return sys.modules[MODULE]


_package()
from ucm_amd import ops  # noqa: E402

DTYPES = {"bfloat16": torch.bfloat16, "float16": torch.float16, "float32": torch.float32}
RHO = 0.95
STEPS = 4            # decode steps a stateful case goes round


# ---------------------------------------------------------------------------------------------- the cases
def listed():
    llama = {"kv_heads": 8, "group": 4, "head_dim": 128}
    bf16 = {"table": "bfloat16", "query": "bfloat16"}
    return [
        # one request of 32768 tokens in one layer: the smallest call an attention hook makes
        {"name": "select_one_request", "op": "select", "layers": 1, "requests": 1, "shortest": 256, "longest": 256, **llama, **bf16},
        # the hook's call for one layer of a ragged batch, float16 model (its representatives are kept widened)
        {"name": "select_one_layer_f16", "op": "select", "layers": 1, "requests": 16, "shortest": 32, "longest": 512, **llama,
         "table": "float32", "query": "float16"},
        # long contexts of a 72B-shaped model, all 80 layers in one launch
        {"name": "select_80_layers", "op": "select", "layers": 80, "requests": 8, "shortest": 512, "longest": 1024,
         "kv_heads": 8, "group": 8, "head_dim": 128, **bf16},
        # a whole decode step: 32 layers of retrieval, then the gather of every selected K and V block
        {"name": "decode_step", "op": "step", "layers": 32, "requests": 16, "shortest": 32, "longest": 512, **llama, **bf16,
         "block_size": 128},
        # end of a prefill of 65536 tokens: the representatives of its blocks in every layer
        {"name": "block_mean_prefill", "op": "mean", "layers": 32, "blocks": 512, "pool": 600, "block_size": 128, "kv_heads": 8,
         "head_dim": 128, "keys": "bfloat16", "table": "bfloat16"},
        # blocks leaving for and coming back from the store
        {"name": "dump_and_load", "op": "moves", "layers": 32, "blocks": 256, "pool": 512, "block_size": 128, "kv_heads": 8,
         "head_dim": 128, "keys": "bfloat16"},
        # end of a prefill with hash codes: token codes, column sums and block codes of 1024 blocks in every layer
        {"name": "hash_encode_prefill", "op": "hash_encode", "layers": 32, "blocks": 1024, "pool": 1100, "block_size": 128,
         "kv_heads": 8, "keys": "bfloat16", "token_codes": True},
        # a decode step by hash codes: 32 requests of 8192-32768 tokens
        {"name": "hash_decode_step", "op": "hash_step", "layers": 32, "requests": 32, "shortest": 64, "longest": 256, "kv_heads": 8,
         "group": 4, "query": "bfloat16"},
        # end of a prefill with KVStar: two-token means of a quarter of the channels
        {"name": "kvstar_repre_prefill", "op": "kvstar_repre", "layers": 32, "blocks": 1024, "pool": 1100, "block_size": 128,
         "merge": 2, "kv_heads": 8, "head_dim": 128, "kept": 32, "keys": "bfloat16"},
        # KVStar's retrieval for every layer of a batch of 16
        {"name": "kvstar_votes_step", "op": "kvstar_votes", "layers": 32, "requests": 16, "shortest": 32, "longest": 512,
         "kv_heads": 8, "group": 4, "head_dim": 128, "kept": 32, "sub_blocks": 64, "tokens": 8},
        # ESA: retrieval and load plan of a batch layer by layer, then the loads of all layers
        {"name": "esa_step", "op": "esa", "layers": 8, "requests": 16, "shortest": 32, "longest": 512, "kv_heads": 8,
         "head_dim": 128, "block_size": 128},
        # GSA with prefetch: selection, hit/miss/free-list round, loads of the missed blocks
        {"name": "prefetch_round", "op": "prefetch", "layers": 8, "requests": 16, "shortest": 64, "longest": 512, **llama, **bf16,
         "block_size": 128},
    ]


def draw(rng):
    def log(lo, hi):
        return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))

    op = rng.choice(["select", "select", "step", "mean", "moves", "hash_encode", "hash_step", "kvstar_repre", "kvstar_votes",
                     "esa", "prefetch"])
    kv = rng.choice([1, 2, 4, 8, 8])
    group = rng.choice([1, 2, 4, 7, 8])
    dim = rng.choice([64, 128, 128])
    half = rng.choice(["bfloat16", "bfloat16", "float16"])
    size = rng.choice([16, 32, 64, 128])
    layers = rng.choice([1, 1, log(2, 80)])
    # segment lengths are drawn between a shortest and a longest one; `room` bounds layers x blocks of a case
    requests, longest = log(1, 64), log(20, 1024)

    def within(room, most_requests=64):
        r = min(requests, most_requests)
        n = max(8, min(longest, room // (layers * r)))
        return {"requests": r, "shortest": max(4, n // rng.choice([1, 2, 8])), "longest": n}

    case = {"op": op, "layers": layers}
    if op == "select":
        table, query = rng.choice([("bfloat16", "bfloat16"), ("float32", "float32"), ("float32", "float16")])
        longest = log(8, 4096)
        case.update(within(250_000), kv_heads=kv, group=group, head_dim=dim, table=table, query=query)
    elif op == "step":
        longest = min(longest, 512)
        case.update(within(2_000_000 // (size * 2)), kv_heads=kv, group=group, head_dim=dim, table="bfloat16", query="bfloat16",
                    block_size=size)
    elif op in ("mean", "hash_encode", "kvstar_repre", "moves"):
        room = {"mean": 32_000, "hash_encode": 24_000, "kvstar_repre": 24_000, "moves": 8_000}[op] * 128 // size
        blocks = log(1, max(1, min(4096, room // layers)))
        case.update(blocks=blocks, pool=blocks + log(1, 64), block_size=size, kv_heads=kv, keys=half)
        if op == "mean":
            case.update(head_dim=dim, table="bfloat16" if half == "bfloat16" else "float32")
        elif op == "hash_encode":
            if size * kv % 32:
                case["block_size"] = 32
            case.update(token_codes=rng.random() < 0.5)
        elif op == "kvstar_repre":
            case.update(head_dim=dim, merge=rng.choice([m for m in (2, 4, 8, 16) if size // m >= 2]), kept=rng.choice([dim // 4, dim]))
        else:
            case.update(head_dim=dim)
    elif op == "hash_step":
        case.update(within(160_000), kv_heads=kv, group=group, query=half)
    elif op == "kvstar_votes":
        tokens = rng.choice([1, 3, 8])
        case.update(within(100_000), kv_heads=kv, group=group, head_dim=dim, kept=rng.choice([dim // 4, dim]),
                    sub_blocks=rng.choice([8, 16, 64]), tokens=tokens)
        if case["sub_blocks"] * case["kept"] > 4096:
            case["sub_blocks"] = 8
    elif op == "esa":
        layers = case["layers"] = min(layers, 8)
        case.update(within(30_000 * 16 // size, 32), kv_heads=kv, head_dim=dim, block_size=size)
    else:
        layers = case["layers"] = min(layers, 8)
        case.update(within(30_000 * 16 // size, 32), kv_heads=kv, group=rng.choice([1, 4, 8]), head_dim=dim, table="bfloat16",
                    query="bfloat16", block_size=size)
        case["longest"] = max(case["longest"], 56)
        case["shortest"] = max(case["shortest"], 50)
    return case


# ---------------------------------------------------------------------------------------------- inputs
def _lengths(case):
    n = np.random.default_rng([case["requests"], case["shortest"], case["longest"]]).integers(
        case["shortest"], case["longest"] + 1, case["requests"]).astype(np.int32)
    n[0] = case["longest"]
    return n


def _topk(lens):
    """3 % of the blocks, at least 16, plus the first one and the last two."""
    return np.maximum(16, (0.03 * lens).astype(np.int32)) + 3


class _Inputs:
    """Everything random about a state, drawn from its seed."""

    def __init__(self, seed):
        self.dev = torch.device("cuda", torch.cuda.current_device())
        self.host = np.random.default_rng(seed)
        self.gen = torch.Generator(device=self.dev)
        self.gen.manual_seed(seed)

    def normal(self, shape, dtype, scale=1.0):
        return torch.empty(shape, dtype=dtype, device=self.dev).normal_(0.0, scale, generator=self.gen)

    def i32(self, a):
        return torch.tensor(np.asarray(a), dtype=torch.int32, device=self.dev)

    def zeros(self, shape, dtype=torch.int32):
        return torch.zeros(shape, dtype=dtype, device=self.dev)

    def drifting(self, shape, dtype):
        """STEPS consecutive decode queries."""
        q, out = self.normal(shape, torch.float32), []
        for _ in range(STEPS):
            out.append(q.to(dtype))
            q = RHO * q + (1.0 - RHO * RHO) ** 0.5 * self.normal(shape, torch.float32)
        return out


def _ragged(case, x):
    lens = _lengths(case)
    off = np.concatenate([[0], np.cumsum(lens)[:-1]]).astype(np.int32)
    rows, longest = int(lens.sum()), int(lens.max())
    table = x.host.permutation(rows).astype(np.int32)                 # random cache blocks behind the logical ones
    bt = np.zeros((len(lens), longest), np.int32)
    for r, n in enumerate(lens):
        bt[r, :n] = table[off[r] : off[r] + n]
    return {"lens": lens, "off_h": off, "rows": rows, "longest": longest, "off": x.i32(off), "len": x.i32(lens), "bt": x.i32(bt)}


def _selection_state(case, x, topk, queries=None):
    L, n_req, kv, d = case["layers"], case["requests"], case["kv_heads"], case["head_dim"]
    s = _ragged(case, x)
    s["topk_h"] = topk(s["lens"])
    s["topk"] = x.i32(s["topk_h"])
    s["q"] = queries if queries is not None else x.normal((L, n_req, kv * case["group"], d), DTYPES[case["query"]])
    # representatives are block means: N(0, 1 / block size), 128-token blocks
    s["repre"] = x.normal((L, s["rows"], kv * d), DTYPES[case["table"]], 128.0 ** -0.5)
    s["scores"] = x.zeros((L, s["rows"]), torch.float32)
    s["idx"] = torch.full((L, n_req, s["longest"]), -1, dtype=torch.int32, device=x.dev)
    s["phys"] = torch.full_like(s["idx"], -1)
    s["cnt"], s["tickets"] = x.zeros((L, n_req)), x.zeros((L, n_req))
    s["kv_heads"] = kv
    return s


def _select(s, q):
    if s["longest"] <= 1024:
        ops.score_select(q, s["repre"], s["off"], s["len"], s["topk"], s["longest"], s["kv_heads"], s["scores"], s["idx"], s["cnt"],
                         s["tickets"], block_tables=s["bt"], phys_out=s["phys"], total_blocks=s["rows"])
    else:                               # longer requests take two launches, as in the GSA hook
        ops.score_blocks(q, s["repre"], s["off"], s["len"], s["longest"], s["kv_heads"], s["scores"], total_blocks=s["rows"])
        ops.topk_windows(s["scores"], s["off"], s["len"], s["topk"], s["longest"], s["idx"], s["cnt"], block_tables=s["bt"],
                         phys_out=s["phys"])


def _prepare_select(case, x):
    return _selection_state(case, x, _topk)


def _run_select(s):
    _select(s, s["q"])
    return s["scores"], s["idx"], s["cnt"], s["phys"]


def _prepare_step(case, x):
    L, bs, kv, d = case["layers"], case["block_size"], case["kv_heads"], case["head_dim"]
    s = _selection_state(case, x, _topk)
    s["nb"], s["block_bytes"] = s["rows"], bs * kv * d * 2
    s["caches"] = [x.normal((2, s["nb"], bs, kv, d), torch.bfloat16) for _ in range(L)]
    s["layers"] = ops.LayerPointers(s["caches"])
    region = np.minimum(s["topk_h"], s["lens"])
    s["most"] = int(region.max())
    s["region"] = x.i32(region)
    s["dst_off"] = torch.from_numpy(np.concatenate([[0], np.cumsum(region.astype(np.int64) * L * 2)[:-1]]).astype(np.int64)).to(x.dev)
    s["staged"] = int(region.astype(np.int64).sum()) * L * 2
    s["staging"] = torch.zeros(s["staged"] * s["block_bytes"] // 2, dtype=torch.bfloat16, device=x.dev)
    return s


def _run_step(s):
    _select(s, s["q"])
    ops.kv_gather_selected(s["layers"], s["nb"] * s["block_bytes"], s["block_bytes"], s["nb"], s["phys"], s["cnt"], s["dst_off"],
                           s["region"], s["most"], s["staging"], s["staged"])
    return s["scores"], s["idx"], s["cnt"], s["phys"], s["staging"]


def _prepare_blocks(case, x, planes):
    """Per-layer caches of `planes` planes (1: keys only, 2: K and V) and a list of their blocks."""
    L, n, nb = case["layers"], case["blocks"], case["pool"]
    shape = (nb, case["block_size"], case["kv_heads"], case.get("head_dim", 128))
    s = {"case": case, "n": n, "nb": nb}
    s["cache"] = x.normal((L, planes) + shape, DTYPES[case["keys"]])
    s["layers"] = ops.LayerPointers([s["cache"][l, 0] if planes == 1 else s["cache"][l] for l in range(L)])
    s["ids"] = x.i32(x.host.permutation(nb)[:n])
    s["slots"] = x.i32(x.host.permutation(n))
    return s


def _prepare_mean(case, x):
    s = _prepare_blocks(case, x, 1)
    s["repre"] = x.zeros((case["layers"], s["n"], case["kv_heads"] * case["head_dim"]), DTYPES[case["table"]])
    return s


def _run_mean(s):
    c = s["case"]
    ops.block_mean(s["layers"], s["ids"], s["slots"], s["repre"], c["block_size"], c["kv_heads"], c["head_dim"], s["nb"],
                   mode=ops.MEAN_BF16_ROUND)
    return s["repre"]


def _prepare_moves(case, x):
    s = _prepare_blocks(case, x, 2)
    s["block_bytes"] = case["block_size"] * case["kv_heads"] * case["head_dim"] * 2
    s["dump_ids"], s["load_ids"] = s["ids"], x.i32(x.host.permutation(s["nb"])[: s["n"]])
    shape = (s["n"], case["layers"], 2, s["block_bytes"] // 2)
    s["dumped"], s["stored"] = x.zeros(shape, DTYPES[case["keys"]]), x.normal(shape, DTYPES[case["keys"]])
    return s


def _run_moves(s):
    args = (s["layers"], s["nb"] * s["block_bytes"], s["block_bytes"], s["nb"])
    ops.kv_gather_blocks(*args, s["dump_ids"], s["dumped"])
    ops.kv_scatter_blocks(*args, s["load_ids"], s["stored"])
    return s["dumped"], s["cache"]


def _prepare_hash_encode(case, x):
    s = _prepare_blocks(case, x, 1)
    L, n, bs, kv = case["layers"], case["blocks"], case["block_size"], case["kv_heads"]
    s["w"] = x.normal((128, 128), torch.float32).to(DTYPES[case["keys"]])
    s["colsum"] = x.zeros((L, n, kv, 128), torch.int16)
    s["codes"] = x.zeros((L, n, kv, 16), torch.uint8)
    s["tokens"] = x.zeros((L, n, bs, kv, 16), torch.uint8) if case["token_codes"] else None
    return s


def _run_hash_encode(s):
    c = s["case"]
    ops.hash_encode_blocks(s["layers"], s["ids"], s["slots"], s["n"], s["w"], c["block_size"], c["kv_heads"], s["nb"], s["colsum"],
                           s["codes"], token_codes=s["tokens"])
    return s["colsum"], s["codes"], s["tokens"]


def _prepare_hash_step(case, x):
    L, n_req, kv, hq = case["layers"], case["requests"], case["kv_heads"], case["kv_heads"] * case["group"]
    s = _ragged(case, x)
    s["kv_heads"], s["n_req"] = kv, n_req
    s["topk"] = x.i32(_topk(s["lens"]))
    s["w"] = x.normal((128, 128), torch.float32).to(DTYPES[case["query"]])
    s["q"] = x.normal((L, n_req, hq, 128), DTYPES[case["query"]])
    # column sums of 128 signs: even numbers of standard deviation 11
    s["colsum"] = (x.normal((L, s["rows"], kv, 128), torch.float32, 5.7).round_() * 2).clamp_(-128, 128).to(torch.int16)
    bits = (s["colsum"] > 0).view(L, s["rows"], kv, 16, 8).to(torch.uint8)
    s["codes"] = (bits << torch.arange(8, dtype=torch.uint8, device=x.dev)).sum(-1, dtype=torch.uint8)
    s["q_codes"], s["q_sum"] = x.zeros((L, n_req, hq, 16), torch.uint8), x.zeros((L, n_req, 128), torch.int16)
    s["qbar"] = x.zeros((L, n_req, kv, 16), torch.uint8)
    s["scores"] = x.zeros((L, s["rows"]), torch.float32)
    s["idx"] = torch.full((L, n_req, s["longest"]), -1, dtype=torch.int32, device=x.dev)
    s["cnt"] = x.zeros((L, n_req))
    return s


def _run_hash_step(s):
    ops.hash_encode_queries(s["q"], s["w"], s["kv_heads"], s["q_codes"], s["q_sum"], s["qbar"], s["n_req"])
    ops.hash_score_blocks(ops.HASH_SCORE_SUM, s["q_sum"], s["qbar"], s["colsum"], s["codes"], s["off"], s["len"], s["rows"], s["scores"])
    ops.topk_windows(s["scores"], s["off"], s["len"], s["topk"], s["longest"], s["idx"], s["cnt"])
    return s["q_codes"], s["q_sum"], s["qbar"], s["scores"], s["idx"], s["cnt"]


def _channels(case, x, lists):
    """A list of kept channels per (list, kv head), ascending; None when all are kept."""
    if case["kept"] == case["head_dim"]:
        return None
    ranks = torch.rand((lists, case["kv_heads"], case["head_dim"]), device=x.dev, generator=x.gen)
    return ranks.topk(case["kept"], dim=-1).indices.sort(dim=-1).values.to(torch.int32).contiguous()


def _padded(kept):
    return (kept + 15) // 16 * 16


def _prepare_kvstar_repre(case, x):
    s = _prepare_blocks(case, x, 1)
    s["pruned"] = _channels(case, x, case["layers"])
    s["table"] = ops.kvstar_table(case["layers"], case["kv_heads"], s["n"], case["block_size"] // case["merge"], _padded(case["kept"]),
                                  x.dev).zero_()
    return s


def _run_kvstar_repre(s):
    c = s["case"]
    ops.kvstar_block_repre(s["layers"], s["ids"], s["slots"], s["table"], c["block_size"], c["kv_heads"], c["head_dim"], s["nb"],
                           c["merge"], pruned=s["pruned"])
    return s["table"]


def _prepare_kvstar_votes(case, x):
    L, n_req, kv, hq, d = case["layers"], case["requests"], case["kv_heads"], case["kv_heads"] * case["group"], case["head_dim"]
    lens = _lengths(case)
    rows, longest, n_tasks, pad = int(lens.sum()), int(lens.max()), L * n_req, _padded(case["kept"])
    off = np.concatenate([[0], np.cumsum(lens)[:-1]])
    s = {"case": case, "longest": longest, "tokens": case["tokens"] if case["tokens"] * case["group"] <= 64 else 1, "hq": hq}
    # two-token means of N(0, 1) keys; the channels past `kept` are the table's zero padding
    table = ops.kvstar_table(1, kv, L * rows, case["sub_blocks"], pad, x.dev)[0]
    table.normal_(0.0, 2.0 ** -0.5, generator=x.gen)
    s["table"] = table
    s["q"] = x.normal((n_tasks, s["tokens"], hq, d), torch.float16, 0.25)
    s["q_off"] = torch.arange(n_tasks, dtype=torch.int64, device=x.dev) * (s["tokens"] * hq * d)
    s["off"] = x.i32((off[None, :] + (np.arange(L) * rows)[:, None]).reshape(-1))
    s["len"] = x.i32(np.tile(lens, L))
    s["topk"] = x.i32(np.tile(np.minimum(_topk(lens), lens), L))
    s["pruned"] = _channels(case, x, L)
    s["sel"] = None if s["pruned"] is None else torch.arange(L, dtype=torch.int32, device=x.dev).repeat_interleave(n_req)
    s["ws"] = ops.kvstar_workspace(n_tasks, kv, s["tokens"] * case["group"], longest, case["sub_blocks"], pad, x.dev)
    s["votes"] = x.zeros((L * rows,), torch.float32)
    s["idx"] = torch.full((n_tasks, longest), -1, dtype=torch.int32, device=x.dev)
    s["cnt"] = x.zeros((n_tasks,))
    return s


def _run_kvstar_votes(s):
    ops.kvstar_votes(s["q"], s["q_off"], s["tokens"], s["hq"], s["table"], s["off"], s["len"], s["longest"], s["votes"], s["ws"],
                     d_pruned=s["case"]["kept"], pruned=s["pruned"], pruned_sel=s["sel"])
    ops.kvstar_topk(s["votes"], s["off"], s["len"], s["topk"], s["longest"], s["idx"], s["cnt"])
    ops.kvstar_order(s["votes"], s["off"], s["len"], s["longest"], s["idx"], s["cnt"])
    return s["votes"], s["idx"], s["cnt"]


def _pool_state(s, case, x, cache_blocks):
    """Caches of `cache_blocks` blocks per layer and a pool holding every request's blocks, [block][layer][K|V]."""
    L, bs, kv, d = case["layers"], case["block_size"], case["kv_heads"], case["head_dim"]
    s["nb"], s["block_bytes"] = cache_blocks, bs * kv * d * 2
    s["cache"] = x.zeros((L, 2, cache_blocks, bs, kv, d), torch.bfloat16)
    s["layers"] = ops.LayerPointers([s["cache"][l] for l in range(L)])
    s["pool"] = x.normal((s["rows"], L, 2, bs * kv * d), torch.bfloat16)
    s["pool_block_bytes"] = L * 2 * s["block_bytes"]
    s["at"] = 0


def _next(s):
    s["at"] += 1
    return s["queries"][(s["at"] - 1) % STEPS]


def _prepare_esa(case, x):
    L, n_req, dim = case["layers"], case["requests"], case["kv_heads"] * case["head_dim"]
    s = _ragged(case, x)
    lens = s["lens"]
    topk = np.maximum((0.3 * lens).astype(np.int32), 1)
    most, rows = int(topk.max()), s["rows"]
    _pool_state(s, case, x, int(topk.sum()))
    s["n_layers"], s["most"] = L, most
    s["data"] = x.normal((L, rows, dim), torch.float32, 128.0 ** -0.5)
    s["queries"] = x.drifting((L, n_req, dim), torch.float32)
    slots, src, dst = np.full((L, n_req, s["longest"]), -1), np.full((n_req, s["longest"]), -1), np.full((n_req, most), -1)
    cache_ids, at = x.host.permutation(s["nb"]), 0
    per_layer = [x.host.permutation(rows) for _ in range(L)]
    for r, n in enumerate(lens):
        o = s["off_h"][r]
        for l in range(L):
            slots[l, r, :n] = per_layer[l][o : o + n]
        src[r, :n] = np.arange(o, o + n)
        dst[r, : topk[r]] = cache_ids[at : at + topk[r]]
        at += topk[r]
    s["slots"], s["src"], s["dst"], s["topk"] = x.i32(slots), x.i32(src), x.i32(dst), x.i32(topk)
    s["req_rows"] = torch.arange(n_req, dtype=torch.int32, device=x.dev)
    s["ws"] = torch.empty(n_req * s["longest"], dtype=torch.float32, device=x.dev)
    minus = lambda *shape: torch.full(shape, -1, dtype=torch.int32, device=x.dev)  # noqa: E731
    s["idx"], s["pos"], s["resident"] = minus(L, n_req, most), minus(L, n_req, most), minus(L, n_req, most)
    s["load"], s["slot_of"] = minus(L, n_req, most), minus(L, n_req, most)
    s["best"] = x.zeros((L, n_req, most), torch.float32)
    s["cnt"], s["miss"] = x.zeros((L, n_req)), x.zeros((L, n_req))
    return s


def _run_esa(s):
    q = _next(s)
    for l in range(s["n_layers"]):
        one = slice(l, l + 1)
        ops.esa_retrieve_rows(s["data"][l], q[l], s["slots"][l], s["longest"], s["req_rows"], s["topk"], s["most"], s["ws"],
                              s["idx"][l], s["pos"][l], s["best"][l], s["cnt"][l])
        ops.delta_plan_rows(s["pos"][one], s["pos"][one], s["cnt"][one], s["req_rows"], s["resident"][one], s["load"][one],
                            s["slot_of"][one], s["miss"][one])
    ops.kv_load_planned(s["layers"], 0, 0, s["n_layers"], s["nb"] * s["block_bytes"], s["block_bytes"], s["nb"], s["pool"],
                        s["pool_block_bytes"], s["load"], s["src"], s["dst"], s["req_rows"])
    return s["idx"], s["pos"], s["best"], s["cnt"], s["load"], s["slot_of"], s["miss"], s["cache"]


KEPT_BLOCKS = 49      # cache blocks a sparsified request keeps (48 selected at most, and one more)


def _prepare_prefetch(case, x):
    from ucm_amd.sparse.gsa.prefetch import GSAPrefetchEngineC
    from ucm_amd.sparse.utils import MIN_TOPK_LEN, compute_topk_len

    L, n_req = case["layers"], case["requests"]
    shape = (L, n_req, case["kv_heads"] * case["group"], case["head_dim"])
    s = _selection_state(case, x, lambda lens: np.array([compute_topk_len(int(n)) for n in lens], np.int32),
                         queries=x.drifting(shape, DTYPES[case["query"]]))
    s["queries"] = s["q"]
    _pool_state(s, case, x, n_req * KEPT_BLOCKS)
    width = 64
    s["free"], s["free_len"] = x.zeros((L, n_req, width)), x.zeros((L, n_req))
    s["table"], s["table_len"] = x.zeros((L, n_req, width)), x.zeros((L, n_req))
    engine = GSAPrefetchEngineC(s["free"], s["table"], s["free_len"], s["table_len"], False)
    src = np.full((n_req, s["longest"]), -1)
    cache_ids = x.host.permutation(s["nb"])
    for r, n in enumerate(s["lens"]):
        # the request's first and last blocks are resident; what lies beyond a selection's shortest length is spare
        held = [int(b) for b in cache_ids[r * KEPT_BLOCKS : (r + 1) * KEPT_BLOCKS]]
        logical = list(range(KEPT_BLOCKS - MIN_TOPK_LEN)) + list(range(int(n) - MIN_TOPK_LEN, int(n)))
        engine.set_blocks_map(r, dict(zip(logical, held)), logical)
        spare = sorted(held[: KEPT_BLOCKS - MIN_TOPK_LEN])
        s["free"][:, r, : len(spare)] = x.i32(spare)
        s["free_len"][:, r] = len(spare)
        src[engine.row_of(r), :n] = np.arange(s["off_h"][r], s["off_h"][r] + n)
    s["engine"], s["src"] = engine, x.i32(src)
    s["req_ids"], s["topk_list"] = list(range(n_req)), [int(k) for k in s["topk_h"]]
    return s


def _run_prefetch(s):
    _select(s, _next(s))
    e = s["engine"]
    e.set_blocks_table_info(s["table"], s["table_len"], s["idx"], s["at"])
    e.run_async_prefetch_bs(s["req_ids"], s["topk_list"], s["req_ids"], 0)
    e.load_missing(s["layers"], s["nb"] * s["block_bytes"], s["block_bytes"], s["nb"], s["pool"].view(-1), s["pool_block_bytes"], s["src"])
    return (s["scores"], s["idx"], s["cnt"], s["table"], s["table_len"], s["free"], s["free_len"], e.load_blocks, e.load_count,
            e.miss_idxs, e.miss_count, s["cache"])


_PREPARE = {"select": _prepare_select, "step": _prepare_step, "mean": _prepare_mean, "moves": _prepare_moves,
            "hash_encode": _prepare_hash_encode, "hash_step": _prepare_hash_step, "kvstar_repre": _prepare_kvstar_repre,
            "kvstar_votes": _prepare_kvstar_votes, "esa": _prepare_esa, "prefetch": _prepare_prefetch}
_RUN = {"select": _run_select, "step": _run_step, "mean": _run_mean, "moves": _run_moves, "hash_encode": _run_hash_encode,
        "hash_step": _run_hash_step, "kvstar_repre": _run_kvstar_repre, "kvstar_votes": _run_kvstar_votes, "esa": _run_esa,
        "prefetch": _run_prefetch}


def prepare(case, seed):
    state = _PREPARE[case["op"]](case, _Inputs(int(seed)))
    state["op"] = case["op"]
    return state


def run(state):
    return _RUN[state["op"]](state)


# ---------------------------------------------------------------------------------------------- work and tolerance
def _size(name):
    return 4 if name == "float32" else 2


def work(case):
    op, L = case["op"], case["layers"]
    kv, d = case["kv_heads"], case.get("head_dim", 128)
    flops = 0
    if "requests" in case:
        lens = _lengths(case)
        rows, n_req = int(lens.sum()), case["requests"]
    if op in ("select", "step", "prefetch"):
        picks = int(np.minimum(_topk(lens), lens).sum())
        nbytes = L * (rows * (kv * d * _size(case["table"]) + 4) + n_req * kv * case["group"] * d * _size(case["query"]) + picks * 8)
        if op == "step":
            nbytes += L * picks * 2 * 2 * case["block_size"] * kv * d * 2
        if op == "prefetch":         # about one selected block in ten is missed at this correlation: K and V in, K and V out
            nbytes += L * n_req * 4 * 4 * case["block_size"] * kv * d * 2
    elif op == "mean":
        nbytes = L * case["blocks"] * kv * d * (case["block_size"] * 2 + _size(case["table"]))
    elif op == "moves":
        nbytes = 2 * L * case["blocks"] * 2 * 2 * case["block_size"] * kv * d * 2
    elif op == "hash_encode":
        vectors = L * case["blocks"] * case["block_size"] * kv
        nbytes = vectors * (256 + (16 if case["token_codes"] else 0)) + L * case["blocks"] * kv * (256 + 16)
        flops = 2 * vectors * 128 * 128
    elif op == "hash_step":
        nbytes = L * (rows * (kv * 256 + 4) + n_req * (kv * case["group"] * (256 + 16) + 256 + kv * 16) + int(_topk(lens).sum()) * 4)
        flops = 2 * L * n_req * kv * (case["group"] + 1) * 128 * 128
    elif op == "kvstar_repre":
        nbytes = L * case["blocks"] * kv * (case["block_size"] * d + case["block_size"] // case["merge"] * _padded(case["kept"])) * 2
    elif op == "kvstar_votes":
        tokens = case["tokens"] if case["tokens"] * case["group"] <= 64 else 1
        nbytes = L * (rows * (kv * case["sub_blocks"] * _padded(case["kept"]) * 2 + 4) + n_req * tokens * kv * case["group"] * d * 2)
        flops = 2 * L * rows * case["sub_blocks"] * kv * case["group"] * tokens * case["kept"]
    else:                            # esa: every candidate's row, and about one block in ten of the 30 % selected is loaded
        picks = int(np.maximum((0.3 * lens).astype(np.int32), 1).sum())
        nbytes = L * (rows * (kv * d * 4 + 4) + picks * 5 * 4 + picks // 10 * 4 * case["block_size"] * kv * d * 2)
    return {"bytes": int(nbytes), "flops": int(flops)}


def tolerance(case):
    """Scores are sums in a fixed order, so they, what is selected from them and every byte moved are the same bits.
    KVStar's votes are fp32 sums whose order is free (against the same sums in fp64, 1024 blocks x 64 and x 8 sub-blocks:
    1e-7 of the norm, 6e-7 of a vote at most), and blocks of nearly equal votes may change places."""
    if case["op"] == "kvstar_votes":
        return {"rel": 1e-6, "max": 1e-5, "differ": 0.002}
    return "exact"
