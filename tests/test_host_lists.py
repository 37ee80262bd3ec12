"""Host lists on their way to the device: int_tensor, the index tensors of
PagedTreeCache, and the page owner's runs of pages against page-by-page
bookkeeping."""

import random

import pytest
import torch


# The edges of what one launch carries (896) and the ends of the type.
@pytest.mark.gpu
@pytest.mark.parametrize("count", [0, 1, 255, 256, 257, 895, 896, 897, 1792, 1793, 20000])
def test_int_tensor_holds_the_list(count):
    import branchcraft_torch as bt
    like = torch.empty(1, device="cuda", dtype=torch.float16)
    ends = [-2**31, 2**31 - 1, 0, -1]
    values = (ends + [random.Random(count).randint(-2**31, 2**31 - 1)
                      for _ in range(count)])[:count]
    out = bt.int_tensor(like, values)
    assert out.dtype == torch.int32 and out.device == like.device and out.tolist() == values


@pytest.mark.gpu
def test_int_tensor_refuses_what_does_not_fit():
    import branchcraft_torch as bt
    like = torch.empty(1, device="cuda", dtype=torch.float16)
    for bad in (2**31, -2**31 - 1):
        with pytest.raises(RuntimeError, match="out of range"):
            bt.int_tensor(like, [0, bad])


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["ints", "tuple", "numpy"])
@pytest.mark.parametrize("tokens", [0, 15, 16, 16 * 897 + 3])
def test_commits_through_either_upload(kind, tokens):
    """Plain ints travel in kernel arguments, others by a copy: same pages,
    for a fork whose partial page is cloned and for two requests at once."""
    import numpy as np
    from branchcraft_torch.transaction import PagedTreeCache
    torch.manual_seed(tokens)
    as_kind = {"ints": list, "tuple": tuple, "numpy": lambda p: [np.int64(x) for x in p]}[kind]
    rows = torch.randn(tokens, 2, 64, device="cuda", dtype=torch.float16)
    dk = torch.randn(2, 40, 2, 64, device="cuda", dtype=torch.float16)
    cache = PagedTreeCache(tokens // 16 + 16, 2, 64)
    one = cache.new(rows, rows)
    two = cache.fork(one)
    first, second = [0, 3, 7], list(range(39, 20, -2))
    cache.commit(one, as_kind(first), dk[:1], -dk[:1])
    cache.commit_many([two, one], [as_kind(second), as_kind(first)], dk, -dk)
    for request, tail in ((one, [dk[0, first], dk[1, first]]), (two, [dk[0, second]])):
        pages, length = cache.pages[request], cache.lengths[request]
        for pool, want in ((cache.k, torch.cat([rows, *tail])),
                           (cache.v, torch.cat([rows, *(-x for x in tail)]))):
            got = pool[torch.tensor(pages, device="cuda")].reshape(-1, 2, 64)[:length]
            assert torch.equal(got, want)


class _PageByPage:
    """alloc and release, a page at a time."""

    def __init__(self, owner):
        self.refcount, self.free = list(owner.refcount), list(owner.free)

    def alloc(self):
        page = self.free.pop()
        assert self.refcount[page] == 0
        self.refcount[page] = 1
        return page

    def release(self, page):
        if self.refcount[page] <= 0:
            raise RuntimeError
        self.refcount[page] -= 1
        if self.refcount[page] == 0:
            self.free.append(page)


@pytest.mark.parametrize("seed", range(6))
def test_runs_of_pages_match_single_pages(seed):
    from branchcraft_torch.pages import PageOwner
    rng = random.Random(seed)
    owner = PageOwner(60)
    single = _PageByPage(owner)
    snapshots = []
    for _ in range(200):
        live = list(owner.pages)
        act = rng.choice(["new", "fork", "checkpoint", "rollback", "accept", "commit"])
        if act == "new" and len(owner.free) >= 4:
            request = owner.new(rng.randint(0, 64))
            assert owner.pages[request] == [single.alloc() for _ in owner.pages[request]]
        elif act in ("fork", "checkpoint") and live:
            request = rng.choice(live)
            if act == "checkpoint":
                snapshots.append(owner.checkpoint(request))
            else:
                owner.fork(request)
            for page in owner.pages[request]:
                single.refcount[page] += 1
        elif act in ("rollback", "accept") and snapshots:
            snapshot = snapshots.pop(rng.randrange(len(snapshots)))
            dropped = list(owner.pages[snapshot.request] if act == "rollback"
                           else snapshot.pages)
            getattr(owner, act)(snapshot)
            for page in dropped:
                single.release(page)
        elif act == "commit" and live and len(owner.free) >= 3:
            request = rng.choice(live)
            before = list(owner.pages[request])
            plan = owner.plan_commit(request, rng.randint(1, 20))
            if plan.cow:
                assert plan.cow == (before[-1], single.alloc())
                single.release(before[-1])
            assert owner.pages[request][len(before):] == [
                single.alloc() for _ in owner.pages[request][len(before):]]
        assert (owner.refcount, owner.free) == (single.refcount, single.free)
        owner.check_invariants()


def test_runs_of_pages_stop_where_single_pages_do():
    """A page already at zero, or a referenced page on the free list: raised
    at that page, with the ones before it done."""
    from branchcraft_torch.pages import PageOwner
    owner = PageOwner(4)
    snapshot = owner.checkpoint(owner.new(48))
    owner.refcount = [2, 0, 2, 0]
    with pytest.raises(RuntimeError, match="page 1 released more often"):
        owner.rollback(snapshot)
    assert owner.refcount == [1, 0, 2, 0] and owner.free == [3] and snapshot.active
    owner = PageOwner(4)
    owner.refcount[1] = 1
    with pytest.raises(RuntimeError, match="free list holds referenced page 1"):
        owner.new(48)
    assert owner.refcount == [1, 1, 0, 0] and owner.free == [3, 2]


@pytest.mark.parametrize("device", ["cuda", "cpu", "meta"])
def test_transaction_on_fake_tensors(device):
    """Shapes of a whole transaction without memory, and for device "cuda"
    without a GPU; no warning about a fake tensor's address."""
    import warnings

    from torch._subclasses.fake_tensor import FakeTensorMode
    from branchcraft_torch.transaction import PagedTreeCache
    with FakeTensorMode(), warnings.catch_warnings():
        warnings.simplefilter("error")

        def half(*shape):
            return torch.empty(shape, device=device, dtype=torch.float16)

        cache = PagedTreeCache(20, 2, 64, device=device)
        one = cache.new(half(19, 2, 64), half(19, 2, 64))
        two = cache.fork(one)
        dk = half(1, 3, 2, 64)
        parent = torch.zeros((1, 3), device=device, dtype=torch.int32)
        out = cache.verify(one, half(1, 3, 4, 64), dk, dk, parent)
        assert out.shape == (1, 3, 4, 64) and out.dtype == torch.float32
        assert cache.commit(one, [0, 2], dk, dk).cow == (1, 2)
        assert cache.commit_many([two, one], [[1], [0]], dk.expand(2, 3, 2, 64),
                                 dk.expand(2, 3, 2, 64))[0].cow is None
        assert cache.lengths == {one: 22, two: 20}
