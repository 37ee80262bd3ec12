"""The calls a serving program makes on this framework, as measurable cases.

A case is one call, or one short sequence of calls, through the public Python
API (``branchcraft_torch``): decode over the packed and the paged cache, tree
verification, and the copy-on-write transaction that admits prompts and
commits accepted tokens.  ``listed()`` names the usual ones, ``draw()`` gives
others of the same ranges.

Sizes are the framework's own: the benchmark's five configurations, the
batch, context and head layouts of the decode and tree sweeps, and the head
layouts of the random-shape tests.
"""

from __future__ import annotations

import math
import random
import sys
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path.cwd() / "branchcraft-cuda_amd" / "python"))

import branchcraft_torch as bt  # noqa: E402
from branchcraft_torch.transaction import PagedTreeCache  # noqa: E402

PAGE = 16
# Query heads, KV heads: GQA groups 1, 2, 4, 7 and 8, and few or many KV heads.
HEADS = ((32, 8), (32, 32), (28, 4), (16, 2), (8, 1), (64, 8), (32, 4), (16, 16), (8, 8), (24, 8))
# No drawn case reads more than the largest listed decode or multiplies more
# than the largest listed tree.
MOST_BYTES = 539e6
MOST_FLOPS = 68e9


def listed():
    return [
        # One request's decode step in the paged cache, short context: launch
        # and latency count, nothing else.
        dict(name="paged 1x512", kind="paged", batch=1, lo=512, hi=512, hq=32, hkv=8, d=128, mix=1),
        # A few very long contexts: one decode step that streams half a GB.
        dict(name="paged 4x16k-32k", kind="paged", batch=4, lo=16384, hi=32768, hq=32, hkv=8, d=128, mix=4),
        # The ordinary decode step of a serving engine: a ragged batch over a
        # block pool of 20000 blocks.
        dict(name="packed 64x128-4096", kind="packed", layout="blocks", pool=20000, batch=64, lo=128,
             hi=4096, hq=32, hkv=8, d=128, mix=5),
        # One long document with nothing else in the batch.
        dict(name="packed 1x32768", kind="packed", layout="blocks", pool=0, batch=1, lo=32768, hi=32768,
             hq=32, hkv=8, d=128, mix=6),
        # Many short chats of a small-head model, in the head-major cache view.
        dict(name="packed 512x16-512 d64", kind="packed", layout="hnd", pool=0, batch=512, lo=16, hi=512,
             hq=32, hkv=8, d=64, mix=7),
        # One request's candidate tree over its prefix.
        dict(name="tree 1x2048x7", kind="tree", batch=1, lo=2048, hi=2048, shared=True, nodes=7,
             parents="random", hq=32, hkv=8, d=128, mix=2),
        # Eight branches forked from one prefix, verified together.
        dict(name="tree 8x2053x7 shared", kind="tree", batch=8, lo=2053, hi=2053, shared=True, nodes=7,
             parents="random", hq=32, hkv=8, d=128, mix=3),
        # A serving batch of unrelated requests with ragged prefixes, each
        # verifying a small tree: the speculative step of an ordinary batch.
        dict(name="tree 64x128-4096x7", kind="tree", batch=64, lo=128, hi=4096, shared=False, nodes=7,
             parents="random", hq=32, hkv=8, d=128, mix=8),
        # Middle-sized trees, an odd node count and a group of seven heads.
        dict(name="tree 16x300-3000x33 d64", kind="tree", batch=16, lo=300, hi=3000, shared=False, nodes=33,
             parents="random", hq=28, hkv=4, d=64, mix=9),
        # The widest trees the API takes: the path is a contraction here.
        dict(name="tree 8x2048x256", kind="tree", batch=8, lo=2048, hi=2048, shared=True, nodes=256,
             parents="random", hq=32, hkv=8, d=128, mix=10),
        # A speculative step through the transaction: eight forks of one
        # prompt are checkpointed and verified, their accepted paths
        # committed (copy-on-write of the shared last page), and the branch
        # taken back.
        dict(name="step 8x2053x7", kind="step", batch=8, lo=2053, hi=2053, nodes=7, accepted=3,
             parents="random", hq=32, hkv=8, d=128, mix=11),
        # A finished prefill's K and V enter the paged pool.
        dict(name="admit 4093", kind="admit", batch=1, lo=4093, hi=4093, hq=32, hkv=8, d=128, mix=12),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    while True:
        kind = rng.choice(("packed", "packed", "paged", "paged", "tree", "tree", "tree", "tree", "step", "admit"))
        hq, hkv = rng.choice(HEADS)
        c = dict(kind=kind, hq=hq, hkv=hkv, d=rng.choice((64, 128)), mix=rng.randrange(1 << 20))
        if kind in ("packed", "paged"):
            c["batch"] = _log_int(rng, 1, 512)
            c["hi"] = _log_int(rng, 33, 32768)
            c["lo"] = c["hi"] if rng.random() < 0.3 else max(1, c["hi"] // rng.choice((2, 8, 32)))
            if kind == "packed":
                c["layout"], c["pool"] = rng.choice(("blocks", "hnd", "nhd")), 0
        elif kind == "tree":
            c["batch"] = _log_int(rng, 1, 64)
            c["hi"] = _log_int(rng, 33, 8192)
            c["shared"] = rng.random() < 0.4
            c["lo"] = c["hi"] if c["shared"] else max(1, c["hi"] // rng.choice((1, 2, 8, 32)))
            c["nodes"] = _log_int(rng, 1, 256)
            c["parents"] = rng.choice(("random", "random", "chain"))
        elif kind == "step":
            c["batch"] = rng.randint(1, 8)
            c["lo"] = c["hi"] = _log_int(rng, 33, 2053)
            c["nodes"] = rng.randint(2, 32)
            c["accepted"] = rng.randint(1, min(6, c["nodes"]))
            c["parents"] = "random"
        else:
            c["batch"] = 1
            c["lo"] = c["hi"] = _log_int(rng, 17, 4093)
        w = work(c)
        if w["bytes"] <= MOST_BYTES and w["flops"] <= MOST_FLOPS:
            return c


# ---------------------------------------------------------------------------
# shapes


def _lengths(c):
    r = random.Random(c["mix"])
    if c["kind"] == "tree" and c["shared"] or c["lo"] == c["hi"]:
        return [c["hi"]] * c["batch"]
    return [r.randint(c["lo"], c["hi"]) for _ in range(c["batch"])]


def _parents(c):
    """parent[0] = -1, parent[i] < i: one tree per request."""
    r = random.Random(c["mix"] + 1)
    rows = []
    for _ in range(c["batch"]):
        rows.append([-1] + [i - 1 if c["parents"] == "chain" else r.randrange(i) for i in range(1, c["nodes"])])
    return rows


def _depths(parents):
    out = []
    for row in parents:
        depth = []
        for p in row:
            depth.append(1 if p < 0 else depth[p] + 1)
        out.append(depth)
    return out


def _path(parents, accepted):
    """A root-to-leaf path of the tree, at most `accepted` nodes of it."""
    path, cur = [], len(parents) - 1
    while cur >= 0:
        path.append(cur)
        cur = parents[cur]
    return path[::-1][:accepted]


def _pages(n):
    return -(-n // PAGE)


def work(case):
    c, lengths = case, _lengths(case)
    hq, hkv, d = c["hq"], c["hkv"], c["d"]
    token = 2 * hkv * d * 2  # one token's K and V
    if c["kind"] in ("packed", "paged"):
        tokens, used = sum(lengths), sum(_pages(n) for n in lengths)
        out = 2 if c["kind"] == "packed" else 4
        return {"bytes": tokens * token + c["batch"] * hq * d * (2 + out) + 4 * used + 4 * c["batch"],
                "flops": 4.0 * d * hq * tokens}
    if c["kind"] == "admit":
        return {"bytes": 2 * lengths[0] * token, "flops": 0.0}
    parents = _parents(c)
    n = c["nodes"]
    prefix = lengths[0] if c["kind"] == "step" or c["shared"] else sum(lengths)
    rows = sum(n * length + sum(dep) for length, dep in zip(lengths, _depths(parents)))
    nbytes = (prefix * token + c["batch"] * n * (token + hq * d * (2 + 4) + 4)
              + 4 * c["batch"] * _pages(max(lengths)) + 4 * c["batch"])
    if c["kind"] == "step":
        # Committed rows, and the shared last page cloned for each request.
        tail = PAGE if lengths[0] % PAGE else 0
        rows_moved = sum(len(_path(p, c["accepted"])) + tail for p in parents)
        nbytes += 2 * rows_moved * token
    return {"bytes": nbytes, "flops": 4.0 * d * hq * rows}


# ---------------------------------------------------------------------------
# inputs


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _half(g, *shape):
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float16)


def _int(rows):
    return torch.tensor(rows, dtype=torch.int32).cuda()


def _table(seed, lengths, width, pool, shared):
    """Block table of shuffled page ids; entries past a length are -1."""
    ids = np.random.default_rng(seed).permutation(pool).astype(np.int32)
    table = np.full((len(lengths), width), -1, dtype=np.int32)
    at = 0
    for i, n in enumerate(lengths):
        k = _pages(n)
        table[i, :k] = ids[:k] if shared else ids[at:at + k]
        at += k
    return torch.from_numpy(table).cuda()


def prepare(case, seed):
    c, lengths = case, _lengths(case)
    b, hq, hkv, d = c["batch"], c["hq"], c["hkv"], c["d"]
    g = _gen(seed)
    s = {"kind": c["kind"]}
    if c["kind"] in ("packed", "paged"):
        used = sum(_pages(n) for n in lengths)
        pool = c.get("pool") or used + used // 8 + 7
        s["q"] = _half(g, b, hq, d)
        s["pages"] = _table(seed, lengths, _pages(c["hi"]), pool, False)
        s["lengths"] = _int(lengths)
        if c["kind"] == "paged":
            s["k"], s["v"] = _half(g, pool, PAGE, hkv, d), _half(g, pool, PAGE, hkv, d)
        else:
            if c["layout"] == "blocks":
                s["kv"] = _half(g, pool, 2, PAGE, hkv, d)
            elif c["layout"] == "hnd":
                s["kv"] = _half(g, pool, hkv, PAGE, 2 * d)
            else:
                s["kv"] = _half(g, pool, PAGE, hkv, 2 * d).transpose(1, 2)
            s["out"] = torch.empty_like(s["q"])
            s["scale"] = 1.0 / math.sqrt(d)
        return s
    if c["kind"] == "admit":
        s["cache"] = PagedTreeCache(_pages(lengths[0]) + 8, hkv, d)
        s["k"], s["v"] = _half(g, lengths[0], hkv, d), _half(g, lengths[0], hkv, d)
        return s
    n, parents = c["nodes"], _parents(c)
    if c["kind"] == "step":
        cache = PagedTreeCache(_pages(lengths[0]) + 2 * b + 8, hkv, d)
        first = cache.new(_half(g, lengths[0], hkv, d), _half(g, lengths[0], hkv, d))
        s["cache"] = cache
        s["requests"] = [first] + [cache.fork(first) for _ in range(b - 1)]
        s["paths"] = [_path(p, c["accepted"]) for p in parents]
        s["parent"] = _int(parents)
    else:
        used = _pages(c["hi"]) if c["shared"] else sum(_pages(x) for x in lengths)
        pool = used + 2 * b
        s["k"], s["v"] = _half(g, pool, PAGE, hkv, d), _half(g, pool, PAGE, hkv, d)
        s["pages"] = _table(seed, lengths, _pages(c["hi"]) + 2, pool, c["shared"])
        s["lengths"] = _int(lengths)
        s["parent"] = _int(parents)
    s["q"] = _half(g, b, n, hq, d)
    s["dk"], s["dv"] = _half(g, b, n, hkv, d), _half(g, b, n, hkv, d)
    return s


# ---------------------------------------------------------------------------
# the calls


def run(s):
    kind = s["kind"]
    if kind == "paged":
        return bt.paged_decode(s["q"], s["k"], s["v"], s["pages"], s["lengths"])
    if kind == "packed":
        return bt.packed_decode_out(s["q"], s["kv"], s["pages"], s["lengths"], s["out"], s["scale"])
    if kind == "tree":
        return bt.tree_verify(s["q"], s["k"], s["v"], s["pages"], s["lengths"], s["dk"], s["dv"], s["parent"])
    cache = s["cache"]
    if kind == "admit":
        request = cache.new(s["k"], s["v"])
        # The request ends here: its pages go back, last one first, so that
        # the next prompt takes them in the same order.
        pages = cache.pages.pop(request)
        cache.lengths.pop(request)
        for page in reversed(pages):
            cache.owner.release(page)
        return {"k": cache.k, "v": cache.v, "pages": np.array(pages)}
    q, dk, dv, parent = s["q"], s["dk"], s["dv"], s["parent"]
    snapshots, outs = [], []
    for i, request in enumerate(s["requests"]):
        snapshots.append(cache.checkpoint(request))
        outs.append(cache.verify(request, q[i:i + 1], dk[i:i + 1], dv[i:i + 1], parent[i:i + 1]))
    plans = cache.commit_many(s["requests"], s["paths"], dk, dv)
    for snapshot in reversed(snapshots):
        cache.rollback(snapshot)
    where = [[p.request, page, slot] for p in plans for page, slot in zip(p.dest_pages, p.dest_slots)]
    return {"out": outs, "k": cache.k, "v": cache.v, "where": np.array(where)}


# ---------------------------------------------------------------------------
# what the results have to be


def tolerance(case):
    if case["kind"] == "admit":
        return "exact"
    if case["kind"] == "packed":
        # FP16 results: two correct roundings of one value may be an ulp apart.
        return {"rel": 1e-3, "max": 2e-3}
    # FP32 results of FP16 inputs with FP32 sums.
    return {"rel": 1e-5, "max": 1e-4}


def _attend(q, k, v, mask=None):
    """q [R, G, D] for one KV head's group, k and v [T, D], in 64 bits."""
    r, g, d = q.shape
    scores = q.double().reshape(r * g, d) @ k.double().t().contiguous() / math.sqrt(d)
    if mask is not None:
        scores = scores.reshape(r, g, -1).masked_fill(~mask[:, None, :], -math.inf).reshape(r * g, -1)
    return (torch.softmax(scores, dim=-1) @ v.double().contiguous()).reshape(r, g, d)


def _tree_exact(q, k, v, dk, dv, parent):
    """One request: q [N, Hq, D], prefix k and v [T, Hkv, D], draft [N, Hkv, D]."""
    n, hq, d = q.shape
    hkv, t = k.shape[1], k.shape[0]
    mask = torch.zeros((n, t + n), dtype=torch.bool)
    mask[:, :t] = True
    for node in range(n):
        cur = node
        while cur >= 0:
            mask[node, t + cur] = True
            cur = parent[cur]
    mask = mask.to(q.device)
    q = q.reshape(n, hkv, hq // hkv, d)
    out = [_attend(q[:, h], torch.cat((k[:, h], dk[:, h])), torch.cat((v[:, h], dv[:, h])), mask)
           for h in range(hkv)]
    return torch.stack(out, 1).reshape(n, hq, d)


def exact(case, seed):
    c, lengths = case, _lengths(case)
    s = prepare(case, seed)
    hkv, d = c["hkv"], c["d"]
    if c["kind"] == "admit":
        return None
    if c["kind"] == "step":
        cache, parents, outs = s["cache"], _parents(c), []
        for i, request in enumerate(s["requests"]):
            ids = torch.tensor(cache.pages[request], device="cuda")
            k, v = (x[ids].reshape(-1, hkv, d)[:lengths[i]] for x in (cache.k, cache.v))
            outs.append(_tree_exact(s["q"][i], k, v, s["dk"][i], s["dv"][i], parents[i])[None])
        return {"out": outs, "k": None, "v": None, "where": None}
    rows = []
    for i, n in enumerate(lengths):
        ids = s["pages"][i, :_pages(n)].long()
        if c["kind"] == "packed":
            kv = s["kv"][ids]
            if c["layout"] == "blocks":
                k, v = kv[:, 0], kv[:, 1]
            else:
                k, v = kv[..., :d].transpose(1, 2), kv[..., d:].transpose(1, 2)
        else:
            k, v = s["k"][ids], s["v"][ids]
        k, v = k.reshape(-1, hkv, d)[:n], v.reshape(-1, hkv, d)[:n]
        if c["kind"] == "tree":
            rows.append(_tree_exact(s["q"][i], k, v, s["dk"][i], s["dv"][i], _parents(c)[i]))
        else:
            q = s["q"][i].reshape(1, hkv, -1, d)
            rows.append(torch.cat([_attend(q[:, h], k[:, h], v[:, h])[0] for h in range(hkv)]))
    return torch.stack(rows)
