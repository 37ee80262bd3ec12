"""write_prefix_ and PagedTreeCache.new: a prompt's rows in the pages of a
host-side list, bit for bit what copying page by page leaves."""

import pytest
import torch


def _by_page(cache, rows, pages):
    want = cache.clone()
    for i, p in enumerate(pages):
        n = min(16, rows.shape[0] - 16 * i)
        want[p, :n] = rows[16 * i:16 * i + n]
    return want


def _bits(x):
    return x.contiguous().view(torch.int16)


# Tokens at the edges of a slice (4), a page (16) and the ids one launch
# carries (896 pages), and two launches.
@pytest.mark.gpu
@pytest.mark.parametrize("tokens,hkv,d", [(1, 8, 128), (4, 1, 64), (5, 3, 64), (16, 8, 128),
                                          (17, 8, 64), (333, 5, 128), (896 * 16, 1, 64),
                                          (896 * 16 + 5, 2, 64)])
@pytest.mark.parametrize("form", ["plain", "fused", "heads_first", "unaligned", "expanded"])
def test_write_prefix_matches_page_copies(tokens, hkv, d, form):
    import branchcraft_torch as bt
    torch.manual_seed(tokens + d)
    count = -(-tokens // 16)

    def half(*shape):
        return torch.randn(shape, device="cuda", dtype=torch.float16)

    if form == "fused":  # slices of one qkv projection
        fused = half(tokens, 3, hkv, d)
        k, v = fused[:, 1], fused[:, 2]
    elif form == "heads_first":
        k, v = half(hkv, tokens, d).transpose(0, 1), half(tokens, hkv, d)
    elif form == "unaligned":
        k, v = half(tokens * hkv * d + 1)[1:].view(tokens, hkv, d), half(tokens, hkv, d)
    elif form == "expanded":
        k, v = half(tokens, 1, d).expand(tokens, hkv, d), half(1, hkv, d).expand(tokens, hkv, d)
    else:
        k, v = half(tokens, hkv, d), half(tokens, hkv, d)
    ck, cv = half(count + 3, 16, hkv, d), half(count + 3, 16, hkv, d)
    pages = torch.randperm(count + 3)[:count].tolist()
    want_k, want_v = _by_page(ck, k, pages), _by_page(cv, v, pages)
    bt.write_prefix_(ck, cv, k, v, pages)
    assert torch.equal(_bits(ck), _bits(want_k)) and torch.equal(_bits(cv), _bits(want_v))


@pytest.mark.gpu
def test_new_takes_what_the_op_does_not():
    """V of another type or on the host, a strided last dimension, rows that
    are views of the pool, rows under autograd and an empty prompt."""
    from branchcraft_torch.transaction import PagedTreeCache
    torch.manual_seed(4)

    def check(k, v, store=None):
        store = store or PagedTreeCache(12, 2, 64)
        before_k, before_v = store.k.detach().clone(), store.v.detach().clone()
        pages = store.pages[store.new(k, v)]
        assert torch.equal(_bits(store.k.detach()), _bits(_by_page(before_k, k.detach(), pages)))
        assert torch.equal(_bits(store.v.detach()),
                           _bits(_by_page(before_v, v.detach().to(before_v), pages)))
        return store

    k = torch.randn(37, 2, 64, device="cuda", dtype=torch.float16)
    check(k, torch.randn(37, 2, 64, device="cuda"))
    check(k, torch.randn(37, 2, 64, dtype=torch.float16))
    check(torch.randn(37, 64, 2, device="cuda", dtype=torch.float16).transpose(1, 2), k)
    check(k[:0], k[:0])
    assert check(k.clone().requires_grad_(), k).k.requires_grad
    store = check(k, k)
    check(store.k[:2].view(32, 2, 64), store.v[:2].view(32, 2, 64), store)


def test_new_on_a_host_pool_copies_by_page():
    pytest.importorskip("branchcraft_torch")
    from branchcraft_torch.transaction import PagedTreeCache
    store = PagedTreeCache(5, 2, 64, device="cpu")
    k, v = (torch.randn(19, 2, 64).half() for _ in range(2))
    pages = store.pages[store.new(k, v)]
    assert torch.equal(store.k, _by_page(torch.zeros_like(store.k), k, pages))
    assert torch.equal(store.v, _by_page(torch.zeros_like(store.v), v, pages))


@pytest.mark.parametrize("grad", [False, True])
def test_write_prefix_moves_the_version_counters(grad):
    """Once per call, on the pools alone; fake tensors, so that it runs
    without a GPU.  An inference pool is refused outside inference mode, as
    an in-place copy into it is."""
    import branchcraft_torch as bt
    from torch._subclasses.fake_tensor import FakeTensorMode
    with FakeTensorMode(), torch.set_grad_enabled(grad):
        pools = [torch.zeros(4, 16, 2, 64, device="cuda", dtype=torch.float16) for _ in range(2)]
        rows = [torch.zeros(19, 2, 64, device="cuda", dtype=torch.float16) for _ in range(2)]
        for calls in (1, 2):
            bt.write_prefix_(*pools, *rows, [2, 0])
            assert [x._version for x in pools + rows] == [calls, calls, 0, 0]
        with torch.inference_mode():
            frozen = [x.clone() for x in pools]
            bt.write_prefix_(*frozen, *rows, [2, 0])
        with pytest.raises(RuntimeError, match="inference tensor"):
            bt.write_prefix_(*frozen, *rows, [2, 0])


@pytest.mark.gpu
def test_backward_sees_a_prompt_enter_the_pool():
    """A pool saved for backward before ``new`` has other values after it."""
    from branchcraft_torch.transaction import PagedTreeCache
    store = PagedTreeCache(4, 2, 64)
    rows = torch.randn(19, 2, 64, device="cuda", dtype=torch.float16)
    x = torch.ones((), device="cuda", dtype=torch.float16, requires_grad=True)
    y = (store.k * x).sum()
    store.new(rows, rows)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        y.backward()


@pytest.mark.gpu
def test_page_ids_past_32_bits_are_skipped():
    """As other ids outside the pool: none of them names a page by its low
    bits."""
    import branchcraft_torch as bt
    pools = [torch.zeros(8, 16, 2, 64, device="cuda", dtype=torch.float16) for _ in range(2)]
    rows = torch.randn(16 * 6, 2, 64, device="cuda", dtype=torch.float16)
    pages = [2**32 + 1, 2, -2**32 + 3, 2**63 - 1, -2**63, 8]
    want = torch.zeros_like(pools[0])
    want[2] = rows[16:32]
    bt.write_prefix_(*pools, rows, rows, pages)
    assert all(torch.equal(x, want) for x in pools)


@pytest.mark.gpu
def test_new_under_autograd_is_what_slice_copies_are():
    """A leaf pool is refused, a tracked pool keeps its graph (a row that a
    later prompt overwrites gets no gradient), and a tangent reaches the pool."""
    import torch.autograd.forward_ad as fw
    from branchcraft_torch.transaction import PagedTreeCache
    k = torch.randn(32, 2, 64, device="cuda", dtype=torch.float16)
    store = PagedTreeCache(4, 2, 64)
    store.k.requires_grad_()
    with pytest.raises(RuntimeError, match="leaf Variable"):
        store.new(k, k)
    for tracked in ("k", "v"):
        store, rows = PagedTreeCache(4, 2, 64), k.clone().requires_grad_()
        first = store.new(*((rows, k) if tracked == "k" else (k, rows)))
        for page in reversed(store.pages.pop(first)):
            store.owner.release(page)
        store.new(k[:16], k[:16])  # over the first page
        getattr(store, tracked).sum().backward()
        assert torch.equal(rows.grad[:16], torch.zeros_like(k[:16]))
        assert torch.equal(rows.grad[16:], torch.ones_like(k[16:]))
    for at in range(2):
        with fw.dual_level():
            store = PagedTreeCache(4, 2, 64)
            pair = [k, k]
            pair[at] = fw.make_dual(k, 2 * k)
            store.new(*pair)
            tangents = [fw.unpack_dual(x).tangent for x in (store.k, store.v)]
            assert tangents[1 - at] is None
            assert torch.equal(tangents[at][:2].reshape(32, 2, 64), 2 * k)
