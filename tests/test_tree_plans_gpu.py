"""Tree verification plans of batched and wide trees, at the edges of their
tiles, steps, parts and ranges, against the CPU oracle.

tree_wide_kernel shares K/V tiles between row tiles: two or four a workgroup,
whole or split by the batch's lengths.  tree_flat_kernel walks equal ranges of a
ragged batch's tiles.  Which kernel a call launches follows from its shape (the
workspace's size tells which); whether its shares or ranges are taken, or whole
units behind them, from the lengths (the workspace's last word).  Short lengths
under large page tables keep the oracle cheap and leave shares and ranges uneven
or empty.  The gate is the reference driver's 3e-4 (src/main.cu:505-509).
"""

import numpy as np
import pytest
import torch

import branchcraft_capi as capi
import gpu_helpers as G
from oracle import oracle_np

pytestmark = pytest.mark.gpu

EDGES = [0, 1, 15, 16, 17, 31, 32, 33, 63, 64, 65, 95, 96, 127, 129, 200]


def _case(seed, batch, nodes, hq, hkv, d, max_pages, pool=None, longest=0, parents="random"):
    """Lengths from EDGES in a shuffled order (the first `longest` tokens, if
    given), distinct pages, some of them outside the pool or with NaN past the
    length."""
    rng = np.random.default_rng(seed)
    lengths = np.array([EDGES[i % len(EDGES)] for i in range(batch)], dtype=np.int32)
    rng.shuffle(lengths)
    lengths[0] = max(lengths[0], min(longest, max_pages * 16))
    npg = [-(-int(x) // 16) for x in lengths]
    used = sum(npg) + 1
    pool = max(pool or 0, used)
    ids = rng.permutation(pool).astype(np.int32)
    # Only the pages in use are filled; the rest of a large pool stays zero.
    g = torch.Generator(device="cuda").manual_seed(seed)
    k, v = (torch.zeros((pool, 16, hkv, d), device="cuda", dtype=torch.float16) for _ in range(2))
    live = torch.from_numpy(ids[:used].astype(np.int64)).cuda()
    for t in (k, v):
        t[live] = torch.randn((used, 16, hkv, d), generator=g, device="cuda", dtype=torch.float16)
    pages = np.full((batch, max_pages), -1, dtype=np.int32)
    at = 0
    for b in range(batch):
        pages[b, :npg[b]] = ids[at:at + npg[b]]
        at += npg[b]
        if lengths[b] % 16:
            last = int(pages[b, npg[b] - 1])
            k[last, lengths[b] % 16:] = float("nan")
            v[last, lengths[b] % 16:] = float("inf")
    par = oracle_np.random_parents(rng, batch, nodes)
    if parents == "chain":
        par[:] = np.arange(-1, nodes - 1)
    elif parents == "malformed":  # cycles, self-loops, parents out of range
        par[1 % batch] = (np.arange(nodes) + 1) % nodes
        par[2 % batch] = np.arange(nodes)
        par[3 % batch, nodes // 2:] = nodes + 5
        par[4 % batch, 1:] = -9
    dq, dk, dv = (rng.standard_normal((batch, nodes, h, d)).astype(np.float16)
                  for h in (hq, hkv, hkv))
    return k, v, pages, lengths, dq, dk, dv, par.astype(np.int32)


def _run(fix, workspace, captured=False):
    k, v, pages, lengths, dq, dk, dv, par = fix
    b, n, hq, d = dq.shape
    shape = capi.Shape(b, hq, k.shape[2], d, pages.shape[1], k.shape[0])
    tp, tl, tq, tdk, tdv, tpar = (G.dev(x) for x in (pages, lengths, dq, dk, dv, par))
    out = G.nan_out((b, n, hq, d), 0)
    prefix = capi.Inputs(None, k.data_ptr(), v.data_ptr(), tp.data_ptr(), tl.data_ptr(), None)
    ins = capi.TreeInputs(prefix, tq.data_ptr(), tdk.data_ptr(), tdv.data_ptr(),
                          tpar.data_ptr(), out.data_ptr())
    L = G.lib()
    if workspace:
        nbytes = L.bc_tree_verify_workspace_size(shape, n)
        ws = torch.full((max(1, nbytes),), 0xff, device="cuda", dtype=torch.uint8)  # NaN partials
        G.check(L.bc_tree_verify_ws(shape, ins, n, ws.data_ptr(), nbytes, G.stream()), "ws call")
    elif captured:
        graph = torch.cuda.CUDAGraph()
        torch.cuda.synchronize()
        with torch.cuda.graph(graph):
            G.check(L.bc_tree_verify(shape, ins, n, G.stream()), "captured call")
        replays = []
        for _ in range(3):
            out.fill_(float("nan"))
            graph.replay()
            torch.cuda.synchronize()
            replays.append(out.clone())
        assert all(torch.equal(x, replays[0]) for x in replays)
    else:
        G.check(L.bc_tree_verify(shape, ins, n, G.stream()), "call")
    torch.cuda.synchronize()
    return out.cpu().numpy()


def _check(fix, oracle, splits):
    k, v, pages, lengths, dq, dk, dv, par = fix
    b, n, hq, d = dq.shape
    shape = capi.Shape(b, hq, k.shape[2], d, pages.shape[1], k.shape[0])
    assert (G.lib().bc_tree_verify_workspace_size(shape, n) > 0) == splits
    # The oracle sees the pages in use only, renumbered.
    live = np.unique(pages[pages >= 0])
    small = np.searchsorted(live, np.maximum(pages, live[0] if len(live) else 0)).astype(np.int32)
    small[pages < 0] = -1
    pick = torch.from_numpy(live.astype(np.int64)).cuda()
    expected = oracle.tree(k[pick].cpu().numpy(), v[pick].cpu().numpy(), small, lengths, dq, dk,
                           dv, par, threads=16)
    for workspace in (True, False):
        G.gate(_run(fix, workspace), expected, 3e-4, f"workspace={workspace}")


@pytest.mark.parametrize("batch,nodes,hq,hkv,d,max_pages,splits,parents", [
    (28, 24, 32, 8, 128, 14, False, "random"),    # three row tiles: an idle wave
    (28, 32, 32, 8, 128, 14, False, "malformed"),  # four, exactly full
    (28, 33, 32, 8, 128, 14, False, "chain"),     # five: a group of one; two draft tiles
    (32, 100, 28, 4, 64, 14, False, "random"),    # group 7: 22 row tiles, partly filled rows
    (7, 256, 32, 8, 128, 14, False, "chain"),     # the widest tree: eight draft tiles
    (2, 256, 64, 8, 64, 14, False, "malformed"),
    # Draft tiles that no row of a row group sees: a group of 128 nodes, one
    # with its last ancestors in the first tile of a window, and odd counts.
    (40, 256, 8, 8, 64, 14, False, "random"),
    (40, 129, 8, 8, 128, 14, False, "malformed"),
    (28, 97, 28, 4, 128, 60, False, "chain"),
    (28, 65, 32, 8, 128, 58, False, "random"),
    # The same past 64 page ids: registers that move up by the tiles left out
    # and are loaded again, at both head dimensions.
    (28, 100, 28, 4, 128, 130, False, "random"),
    (40, 200, 8, 8, 64, 130, False, "chain"),
    (64, 9, 32, 8, 64, 14, False, "random"),      # two row tiles, two workgroups per CU
    (32, 16, 32, 8, 128, 60, False, "malformed"),  # two, one workgroup per CU
    # The ancestor sets of one wave: 64 nodes, one short of them, chains and
    # cycles over all of them.
    (30, 64, 32, 8, 128, 14, False, "chain"),
    (30, 63, 32, 8, 64, 14, False, "malformed"),
    (30, 64, 32, 8, 64, 14, False, "malformed"),
    # Tables that have room for shares, over lengths that mostly do not fill
    # them (test_routes_follow_the_lengths has both sides).
    (20, 16, 32, 8, 128, 130, True, "random"),
    (32, 16, 32, 8, 128, 130, True, "chain"),
    (140, 9, 8, 1, 128, 130, True, "malformed"),  # requests in three windows of 64
    (250, 16, 4, 1, 128, 130, True, "random"),    # in four; more requests than shares to spare
    (12, 128, 16, 4, 64, 130, True, "chain"),     # shares that begin between draft tiles
    (32, 64, 16, 16, 64, 130, False, "random"),   # D = 64: 512 groups, whole
    (16, 64, 16, 16, 64, 130, True, "random"),
    (16, 33, 28, 4, 64, 190, True, "random"),     # four row tiles a workgroup
    (8, 64, 32, 8, 128, 190, True, "chain"),      # more than a scratch slot holds
    (28, 40, 16, 4, 64, 190, True, "random"),     # an even batch but for one long request
])
def test_wide_trees(batch, nodes, hq, hkv, d, max_pages, splits, parents, oracle):
    fix = _case(batch + nodes, batch, nodes, hq, hkv, d, max_pages, parents=parents,
                longest=1500 if max_pages > 100 else 0)
    _check(fix, oracle, splits)


@pytest.mark.parametrize("batch,nodes,hq,hkv,d,max_pages,pool,parents", [
    (9, 32, 32, 4, 128, 226, 2040, "random"),   # a pool past the L2s
    (6, 12, 24, 8, 128, 136, 800, "chain"),     # two row tiles
    (21, 16, 28, 4, 64, 147, 3080, "malformed"),
    (3, 33, 64, 8, 128, 165, 520, "random"),    # nine row tiles
    (9, 32, 32, 4, 128, 226, 0, "chain"),       # the same shape, a small pool: whole, a row tile each
])
def test_wide_trees_over_large_pools(batch, nodes, hq, hkv, d, max_pages, pool, parents, oracle):
    fix = _case(batch + nodes, batch, nodes, hq, hkv, d, max_pages, pool=pool, parents=parents,
                longest=2000)
    _check(fix, oracle, pool > 0)


@pytest.mark.parametrize("batch,nodes,hq,hkv,d,max_pages", [
    (12, 128, 16, 4, 64, 130),  # few wide units: a row tile a workgroup
    (32, 16, 32, 8, 128, 130),  # one per CU: whole wide units
])
def test_split_shapes_under_capture(batch, nodes, hq, hkv, d, max_pages, oracle):
    """A captured call without a workspace has no scratch and runs whole units."""
    fix = _case(3, batch, nodes, hq, hkv, d, max_pages, longest=1500)
    k, v, pages, lengths, dq, dk, dv, par = fix
    expected = oracle.tree(k.cpu().numpy(), v.cpu().numpy(), pages, lengths, dq, dk, dv, par,
                           threads=16)
    G.gate(_run(fix, False, captured=True), expected, 3e-4, "captured")


@pytest.mark.parametrize("batch,nodes,hq,hkv,d,max_pages,pool,longest,parents", [
    (64, 7, 32, 8, 128, 128, 2048, 2048, "random"),
    (50, 1, 32, 8, 128, 129, 2048, 0, "random"),     # one node: one-tile units
    (64, 32, 8, 8, 128, 128, 2048, 700, "malformed"),  # a full draft tile
    (130, 8, 8, 2, 128, 200, 8192, 3200, "random"),  # lengths in several windows of 64
    (64, 31, 16, 16, 64, 128, 2048, 1000, "chain"),  # 31 draft tokens
    (300, 4, 7, 1, 128, 200, 16384, 2000, "random"),  # more requests than ranges
])
def test_flat_ranges(batch, nodes, hq, hkv, d, max_pages, pool, longest, parents, oracle):
    fix = _case(batch + nodes, batch, nodes, hq, hkv, d, max_pages, pool=pool, longest=longest,
                parents=parents)
    _check(fix, oracle, True)


def test_pages_outside_the_pool_are_skipped(oracle):
    """Ids past the pool and negative ones inside a length, on the wide kernel
    (whole units and shares), the flat one and the single pass behind them: the
    result is the one without those pages' tokens."""
    for shape in ((28, 32, 32, 8, 128, 14, None, 0, None), (64, 7, 32, 8, 128, 128, 2048, 0, False),
                  (64, 7, 32, 8, 128, 128, 2048, 2048, True),
                  (8, 64, 32, 8, 128, 190, None, 3000, True),
                  (16, 33, 28, 4, 64, 190, None, 3000, True),
                  (16, 16, 32, 8, 128, 130, 2048, 0, False)):
        batch, nodes, hq, hkv, d, max_pages, pool, longest, in_shares = shape
        k, v, pages, lengths, dq, dk, dv, par = _case(5, batch, nodes, hq, hkv, d, max_pages,
                                                      pool=pool, longest=longest)
        full = [b for b in range(batch) if lengths[b] >= 64]
        bad = pages.copy()
        cut, cut_len = np.full_like(pages, -1), lengths.copy()
        for b in range(batch):
            row = list(pages[b, :-(-int(lengths[b]) // 16)])
            if b in full:
                bad[b, 1] = k.shape[0] + 3 if b % 2 else -1
                del row[1]
                cut_len[b] -= 16
            cut[b, :len(row)] = row
        if in_shares is not None:
            assert _cuts((k, v, bad, lengths, dq, dk, dv, par)) == in_shares
        live = torch.from_numpy(np.unique(cut[cut >= 0]).astype(np.int64)).cuda()
        ren = np.full(k.shape[0], -1, dtype=np.int32)
        ren[live.cpu().numpy()] = np.arange(len(live))
        small = np.where(cut >= 0, ren[np.maximum(cut, 0)], -1).astype(np.int32)
        expected = oracle.tree(k[live].cpu().numpy(), v[live].cpu().numpy(), small, cut_len, dq,
                               dk, dv, par, threads=16)
        for workspace in (True, False):
            got = _run((k, v, bad, lengths, dq, dk, dv, par), workspace)
            G.gate(got, expected, 3e-4, f"{shape} workspace={workspace}")


def _cuts(fix):
    """Whether a workspace call took its units in shares or ranges: the
    workspace's last word.  Whole units leave no partials (the records stand in
    the final 4 KB)."""
    k, v, pages, lengths, dq, dk, dv, par = fix
    b, n, hq, d = dq.shape
    shape = capi.Shape(b, hq, k.shape[2], d, pages.shape[1], k.shape[0])
    tp, tl, tq, tdk, tdv, tpar = (G.dev(x) for x in (pages, lengths, dq, dk, dv, par))
    out = G.nan_out((b, n, hq, d), 0)
    ins = capi.TreeInputs(
        capi.Inputs(None, k.data_ptr(), v.data_ptr(), tp.data_ptr(), tl.data_ptr(), None),
        tq.data_ptr(), tdk.data_ptr(), tdv.data_ptr(), tpar.data_ptr(), out.data_ptr())
    L = G.lib()
    nbytes = L.bc_tree_verify_workspace_size(shape, n)
    ws = torch.full((nbytes,), 0xff, device="cuda", dtype=torch.uint8)
    G.check(L.bc_tree_verify_ws(shape, ins, n, ws.data_ptr(), nbytes, G.stream()), "ws call")
    torch.cuda.synchronize()
    taken = int(ws[-4:].view(torch.int32))
    assert taken in (0, 1) and (taken or bool((ws[:-4096] == 0xff).all()))
    return bool(taken)


def _workspace(route, batch, d):
    """Bytes of a route's partials, (max, sum) pairs, records and last word."""
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    rows, records = {"flat": (2 * cus * 32, cus), "wide2": (2 * cus * 64, batch),
                     "wide4": (2 * cus * 128, batch)}[route]
    return rows * (d * 4 + 8) + records * 8 + 4


@pytest.mark.parametrize("route,batch,nodes,hq,hkv,d,max_pages,pool,longest,parents,cut", [
    # Tables of 4096 tokens and more over short lengths: whole units, two
    # requests a workgroup or one.
    ("flat", 64, 7, 32, 8, 128, 258, 2048, 0, "random", False),
    ("flat", 33, 8, 32, 8, 64, 800, 4096, 0, "malformed", False),
    ("flat", 7, 16, 16, 8, 128, 1024, 2048, 200, "chain", False),
    ("wide4", 8, 33, 32, 8, 128, 258, 0, 0, "random", False),
    ("wide4", 1, 256, 32, 8, 128, 512, 0, 300, "malformed", False),
    ("wide2", 16, 16, 32, 8, 128, 258, 2048, 0, "chain", False),
    ("wide4", 16, 33, 28, 4, 64, 258, 2048, 500, "random", False),
    ("wide2", 15, 10, 24, 4, 64, 800, 4096, 0, "random", False),  # an odd batch
    # One request far longer than its equal part: cut.
    ("flat", 50, 1, 32, 8, 128, 129, 2048, 2064, "random", True),      # one-tile units
    ("flat", 64, 32, 8, 8, 128, 128, 2048, 2048, "malformed", True),   # a full draft tile
    ("flat", 64, 31, 16, 16, 64, 250, 2048, 4000, "chain", True),      # 31 draft tokens
    ("flat", 300, 4, 7, 1, 128, 200, 16384, 3200, "random", True),     # more requests than ranges
    ("flat", 130, 8, 8, 2, 128, 200, 8192, 3200, "random", True),      # three windows of 64
    ("wide2", 20, 16, 32, 8, 128, 160, 0, 2560, "random", True),
    ("wide4", 140, 9, 8, 1, 128, 160, 0, 2560, "malformed", True),     # three windows of 64
    ("wide2", 250, 16, 4, 1, 128, 160, 0, 2500, "random", True),       # nearly every slot
    ("wide4", 12, 33, 28, 4, 64, 190, 2048, 3040, "random", True),
    ("wide4", 4, 64, 32, 8, 128, 190, 2048, 3000, "chain", True),      # many shares, four rows a wave
    ("wide2", 3, 9, 32, 8, 128, 250, 2048, 4000, "random", True),
    # Two units per CU and more (D = 64: past two): at any length.
    ("wide4", 8, 64, 32, 8, 128, 190, 0, 0, "malformed", True),
    ("wide4", 12, 128, 16, 4, 64, 130, 0, 0, "chain", True),
    ("wide4", 32, 16, 64, 4, 128, 130, 0, 0, "random", True),
])
def test_routes_follow_the_lengths(route, batch, nodes, hq, hkv, d, max_pages, pool, longest,
                                   parents, cut, oracle):
    """The table's width only says that a batch may be long."""
    fix = _case(batch + nodes, batch, nodes, hq, hkv, d, max_pages, pool=pool, longest=longest,
                parents=parents)
    shape = capi.Shape(batch, hq, hkv, d, max_pages, fix[0].shape[0])
    assert G.lib().bc_tree_verify_workspace_size(shape, nodes) == _workspace(route, batch, d)
    assert _cuts(fix) == cut
    _check(fix, oracle, True)


def test_whole_units_do_not_depend_on_the_table():
    """A short batch under a wide table over a large pool takes the tight
    table's single pass, bit for bit, also when its neighbours are longer."""
    k, v, pages, lengths, dq, dk, dv, par = _case(9, 64, 7, 32, 8, 128, 14)
    tight = _run((k, v, pages, lengths, dq, dk, dv, par), True)
    big_k, big_v = (torch.zeros((2048, *x.shape[1:]), device="cuda", dtype=x.dtype) for x in (k, v))
    big_k[:k.shape[0]], big_v[:v.shape[0]] = k, v
    wide = np.full((64, 512), -1, dtype=np.int32)
    wide[:, :pages.shape[1]] = pages
    assert np.array_equal(_run((big_k, big_v, wide, lengths, dq, dk, dv, par), True), tight)


@pytest.mark.parametrize("batch,nodes,hq,hkv,d,max_pages,pool", [
    (64, 7, 32, 8, 128, 128, 2048),  # ranges
    (16, 16, 32, 8, 128, 160, 2048),  # shares of two row tiles
    (12, 33, 28, 4, 64, 190, 2048),   # of four
])
def test_a_captured_call_follows_the_lengths(batch, nodes, hq, hkv, d, max_pages, pool):
    """One graph, replayed over lengths that are cut, left whole and cut again:
    each time the eager call's bits."""
    k, v, pages, lengths, dq, dk, dv, par = _case(3, batch, nodes, hq, hkv, d, max_pages, pool=pool,
                                                  longest=16 * max_pages)
    b, n = batch, nodes
    shape = capi.Shape(b, hq, hkv, d, max_pages, k.shape[0])
    tp, tl, tq, tdk, tdv, tpar = (G.dev(x) for x in (pages, lengths, dq, dk, dv, par))
    short = np.minimum(lengths, 70).astype(np.int32)
    L = G.lib()
    nbytes = L.bc_tree_verify_workspace_size(shape, n)
    ws = torch.full((nbytes,), 0xff, device="cuda", dtype=torch.uint8)
    out = G.nan_out((b, n, hq, d), 0)

    def call():
        prefix = capi.Inputs(None, k.data_ptr(), v.data_ptr(), tp.data_ptr(), tl.data_ptr(), None)
        ins = capi.TreeInputs(prefix, tq.data_ptr(), tdk.data_ptr(), tdv.data_ptr(),
                              tpar.data_ptr(), out.data_ptr())
        G.check(L.bc_tree_verify_ws(shape, ins, n, ws.data_ptr(), nbytes, G.stream()), "call")

    eager = {}
    for name, lens in (("long", lengths), ("short", short)):
        tl.copy_(torch.from_numpy(lens))
        call()
        torch.cuda.synchronize()
        eager[name] = (out.clone(), int(ws[-4:].view(torch.int32)))
    assert (eager["long"][1], eager["short"][1]) == (1, 0)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call()
    for name in ("long", "short", "long", "short", "short", "long"):
        tl.copy_(torch.from_numpy(lengths if name == "long" else short))
        out.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager[name][0]), name
