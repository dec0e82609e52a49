"""The cache manager: no page lost, held twice or freed twice, under random orders
of requests; windows give pages back; state slots are exclusive (CPU)."""
import random

import pytest

from hfee_amd.cache import CacheError, CacheGroupSpec, CacheManager, OutOfPages, PagePool

FULL = CacheGroupSpec("full", (2, 2, 16), cache_layers=(0, 1))
WIN = CacheGroupSpec("window", (2, 2, 16), cache_layers=(2,), window=40)


def test_pool_refuses_double_free_and_foreign_free():
    p = PagePool(3)
    a, b = p.take("x"), p.take("y")
    assert (a, b) == (0, 1) and p.num_free == 1
    p.give_back(a, "x")
    with pytest.raises(CacheError, match="freed twice"):
        p.give_back(a, "x")
    with pytest.raises(CacheError, match="belongs to"):
        p.give_back(b, "x")
    assert p.take("z") == a, "the page freed last is handed out first"
    p.take("z")
    with pytest.raises(OutOfPages):
        p.take("z")


def test_reserve_commit_release_and_reuse():
    m = CacheManager([FULL], 16, 6, max_requests=2)
    a = m.admit("a")
    assert m.pages_needed("a", 17) == [2]
    m.reserve("a", 17)
    m.commit("a", 17)
    assert a.length == 17 and m.pages_needed("a", 15) == [0] and m.pages_needed("a", 16) == [1]
    m.admit("b")
    with pytest.raises(OutOfPages):
        m.reserve("b", 16 * 4 + 1)
    assert m.free_pages() == [4], "a failed reservation takes nothing"
    m.reserve("b", 64)
    with pytest.raises(CacheError, match="beyond the reserved pages"):
        m.commit("a", 16)
    with pytest.raises(CacheError, match="state slots"):
        m.admit("c")
    held = list(m.block_table("a", 0))
    m.release("a")
    m.check()
    c = m.admit("c")
    assert c.slot == a.slot
    m.reserve("c", 20)
    assert sorted(m.block_table("c", 0)) == sorted(held), "released pages are used again"
    with pytest.raises(CacheError, match="not live"):
        m.release("a")
    m.check()


def test_window_group_gives_back_pages_the_window_has_passed():
    m = CacheManager([FULL, WIN], 16, [32, 12], max_requests=1)
    m.admit("r")
    n = 0
    for portion in (50, 1, 1, 30, 7, 1, 100, 1, 1):
        m.reserve("r", portion)
        m.commit("r", portion)
        n += portion
        m.check()
        full, win = m.block_table("r", 0), m.block_table("r", 1)
        assert all(p >= 0 for p in full) and len(full) == (n + 15) // 16
        first_needed = max(0, n - 40 + 1)
        for b, page in enumerate(win):
            if (b + 1) * 16 <= first_needed:
                assert page == -1, f"block {b} is behind the window and still held"
            else:
                assert page >= 0, f"block {b} is inside the window and gone"
    assert m.free_pages()[1] >= 12 - 4
    m.release("r")
    m.check()
    assert m.free_pages() == [32, 12]


def test_a_group_that_grows_every_few_tokens():
    """One entry every 5 tokens: n tokens hold ceil(n / 5) entries in ceil(ceil(n / 5) / 16) pages; a
    reservation fails as a whole when that group alone has no page left; truncation cuts it back too."""
    every5 = CacheGroupSpec("full", (2, 24), cache_layers=((0, 1),), every=5)
    m = CacheManager([FULL, every5], 16, [40, 3], max_requests=2)
    m.admit("r")
    n = 0
    for portion in (1, 3, 1, 75, 1, 79, 1, 2, 77):
        m.reserve("r", portion)
        m.commit("r", portion)
        n += portion
        m.check()
        entries = (n + 4) // 5
        assert len(m.block_table("r", 0)) == (n + 15) // 16 and len(m.block_table("r", 1)) == (entries + 15) // 16
    assert n == 240 and m.pages_needed("r", 1) == [1, 1] and m.pages_for_tokens(161) == [11, 3]
    m.admit("s")
    with pytest.raises(OutOfPages):
        m.reserve("s", 1)                  # (the tokens' group has pages, the other has none)
    assert m.block_table("s", 0) == [] and m.free_pages() == [25, 0]
    m.truncate("r", 80)
    assert len(m.block_table("r", 0)) == 5 and len(m.block_table("r", 1)) == 1 and m.free_pages() == [35, 2]
    m.reserve("s", 81)
    m.commit("s", 81)
    m.check()
    m.release("r")
    m.release("s")
    assert m.free_pages() == [40, 3]
    with pytest.raises(CacheError):
        CacheGroupSpec("window", (2, 24), cache_layers=(3,), window=8, every=2)
    with pytest.raises(CacheError):
        CacheManager([FULL, every5], 16, [8, 8], max_requests=1, keep_prefixes=True)


@pytest.mark.parametrize("seed", range(8))
def test_random_orders_keep_every_invariant(seed):
    rng = random.Random(seed)
    m = CacheManager([FULL, WIN], 16, [40, 12], max_requests=5)
    live, counter = {}, 0
    for _ in range(600):
        op = rng.random()
        if op < 0.25 and m.num_free_slots:
            counter += 1
            m.admit(counter)
            live[counter] = 0
        elif op < 0.8 and live:
            rid = rng.choice(list(live))
            n = rng.choice([1, 1, 1, 2, 5, 16, 17, 33, 64])
            if m.can_reserve(rid, n):
                m.reserve(rid, n)
                if rng.random() < 0.9:
                    m.commit(rid, n)
                    live[rid] += n
            else:
                with pytest.raises(OutOfPages):
                    m.reserve(rid, n)
        elif op < 0.9 and live:
            rid = rng.choice(list(live))
            if live[rid] and rng.random() < 0.5:
                try:
                    keep = rng.randrange(live[rid] + 1)
                    m.truncate(rid, keep)
                    live[rid] = keep
                except CacheError:
                    pass          # a window group cannot go back past released pages
        elif live:
            rid = rng.choice(list(live))
            m.release(rid)
            del live[rid]
        m.check()
        for rid, n in live.items():
            assert m.get(rid).length == n
    for rid in list(live):
        m.release(rid)
    m.check()
    assert m.free_pages() == [40, 12] and m.num_free_slots == 5


# ------------------------------------------------------- prefixes kept between requests
def keeping(pages=16, requests=4, groups=1):
    specs = [CacheGroupSpec("full", (2, 1, 16), (g,)) for g in range(groups)]
    return CacheManager(specs, 16, pages, requests, keep_prefixes=True)


def run_whole(m, rid, tokens):
    rc = m.admit(rid, tokens)
    m.reserve(rid, len(tokens) - rc.length)
    m.commit(rid, len(tokens) - rc.length)
    return rc


def test_full_pages_of_a_released_request_wait_for_one_that_begins_alike():
    m = keeping(pages=8, groups=2)
    a = list(range(100, 140))                         # 40 tokens: two full pages and a half
    rc = run_whole(m, "a", a)
    pages = [list(t) for t in rc.tables]
    m.release("a", a)
    m.check()
    assert m.num_kept_pages == 2 and m.free_pages() == [8, 8]          # kept pages count as free
    # the same 32 tokens and then others: both pages come back, as this request's own, in every group
    rc = m.admit("b", a[:32] + [7, 8, 9])
    assert rc.length == rc.reused == 32 and [t[:2] for t in rc.tables] == [p[:2] for p in pages]
    assert m.num_kept_pages == 0 and m.pages_needed("b", 3) == [1, 1]
    m.check()
    m.release("b", a[:32])
    # exactly the kept tokens: one token must still be run (runner.go:219), so the second page stays
    rc = m.admit("c", a[:32])
    assert rc.length == 16 and m.num_kept_pages == 1
    m.release("c", a[:16])
    m.check()
    # the first page differs in its last token: nothing is taken, although the second page's own tokens agree
    rc = m.admit("d", a[:15] + [0] + a[16:40])
    assert rc.length == 0 and m.num_kept_pages == 2
    m.release("d")
    # a page is known by everything before it as well: these 16 tokens behind another beginning are another page
    rc = m.admit("e", [1] * 16 + a[16:40])
    assert rc.length == 0
    m.release("e")
    m.check()


def test_kept_pages_give_way_when_pages_are_needed_the_deepest_of_the_oldest_first():
    m = keeping(pages=4)
    a, b = list(range(200, 232)) + [1], list(range(300, 316)) + [1]
    run_whole(m, "a", a)                      # pages 0, 1, 2
    m.release("a", a)                         # two kept
    run_whole(m, "b", b)                      # two more pages
    m.release("b", b)                         # one kept
    assert m.num_kept_pages == 3 and m.free_pages() == [4]
    m.admit("c")
    m.reserve("c", 32)                        # one page is free, the other comes from a's second page
    assert m.num_kept_pages == 2
    m.check()
    assert m.admit("a2", a).length == 16      # a's first page is still there, its second is gone
    assert m.admit("b2", b).length == 16
    m.check()
    m.release("a2"), m.release("b2")
    with pytest.raises(OutOfPages):
        m.reserve("c", 80)                    # five pages: nothing kept is left to give way
    m.release("c", None)
    m.drop_kept()
    assert m.free_pages() == [4] and m.num_kept_pages == 0
    m.check()


def test_the_same_prefix_is_kept_once():
    m = keeping(pages=8)
    a = list(range(50, 83))
    run_whole(m, "a", a)
    m.admit("b")                              # the same tokens run again beside it (nothing was kept yet)
    m.reserve("b", 33), m.commit("b", 33)
    m.release("a", a), m.release("b", a)
    assert m.num_kept_pages == 2 and len(m.pools[0]._free) == 6
    m.check()


@pytest.mark.parametrize("as_array", [False, True])
def test_a_release_may_know_other_tokens_than_the_admission(as_array):
    """What stays behind lies under the tokens that the release names: more than the prompt's, fewer, or others from some
    place on, which must not be found under the prompt's digests."""
    import numpy as np
    give = (lambda t: np.asarray(t)) if as_array else (lambda t: t)
    m = keeping(pages=12)
    prompt = list(range(40, 120))                       # five pages, of which an admission looks at four
    run_whole(m, "a", give(prompt))
    m.release("a", give(prompt))
    rc = m.admit("b", give(prompt))
    assert rc.length == 64
    m.reserve("b", 48), m.commit("b", 48)               # 112 tokens: seven pages
    other = prompt[:40] + list(range(500, 572))         # (another third page)
    m.release("b", give(other))
    m.check()
    assert m.admit("c", give(prompt)).length == 32      # two pages are the prompt's still
    m.release("c", give(prompt[:16]))                   # fewer tokens than it holds: one page stays
    m.check()
    assert m.admit("d", give(other)).length == 16
    m.check()
    m.release("d")


def test_less_than_a_page_is_not_digested():
    """A prompt that fills no page, or just one (its last token has to run), is admitted and released without digests."""
    m = keeping(pages=12)
    run_whole(m, "a", list(range(64)))
    m.release("a", list(range(64)))
    for n in (0, 1, 15, 16):
        assert m.admit("b", list(range(n))).digests is None and m.get("b").length == 0
        m.release("b", list(range(n)))
    assert m.admit("c", list(range(17))).length == 16
    m.release("c")
    m.check()


def test_tokens_that_are_no_numbers_leave_a_request_as_it_was():
    m = keeping(pages=12)
    run_whole(m, "a", list(range(64)))
    m.release("a", list(range(64)))
    rc = m.admit("b", list(range(40)))
    m.reserve("b", 32), m.commit("b", 32)
    for _ in range(2):
        with pytest.raises(OverflowError):
            m.release("b", list(range(40)) + [2 ** 70] * 24)
    assert len(rc.digests.data) == 8 * len(rc.digests.tokens)
    m.release("b", list(range(64)))
    m.check()


def test_prefixes_are_not_kept_where_a_window_has_given_pages_back():
    with pytest.raises(CacheError, match="every cache group keeps every token"):
        CacheManager([CacheGroupSpec("window", (2, 1, 16), (0,), window=32)], 16, 8, 2, keep_prefixes=True)


@pytest.mark.parametrize("seed", range(6))
def test_random_orders_with_kept_prefixes(seed):
    """Requests from a small family of prompts that begin alike come and go in random order on
    few pages.  A model of the memory (what was written where) shows that every position of a
    live request, taken over or written, holds that request's token, and check() that no page
    is lost, held twice or both kept and owned."""
    rng = random.Random(seed)
    ps = 16
    m = keeping(pages=12, requests=3)
    stems = [[rng.randrange(1000) for _ in range(70)] for _ in range(2)]
    content, live, n = {}, {}, 0          # (page, slot) -> token; rid -> its tokens
    reused = 0
    for _ in range(400):
        if live and (len(live) == 3 or rng.random() < 0.4):
            rid = rng.choice(sorted(live))
            rc = m.get(rid)
            assert [content[(rc.tables[0][p // ps], p % ps)] for p in range(rc.length)] == live[rid][:rc.length]
            m.release(rid, live[rid] if rng.random() < 0.8 else None)
            del live[rid]
        else:
            stem = rng.choice(stems)
            tokens = stem[:rng.randrange(1, 70)] + [rng.randrange(1000) for _ in range(rng.randrange(0, 20))]
            rid, n = n, n + 1
            rc = m.admit(rid, tokens)
            assert rc.length % ps == 0 and rc.length < len(tokens)
            reused += rc.length
            try:
                m.reserve(rid, len(tokens) - rc.length)
            except OutOfPages:
                m.release(rid, tokens)            # only what it took over can stay behind
                m.check()
                continue
            for p in range(rc.length, len(tokens)):
                content[(rc.tables[0][p // ps], p % ps)] = tokens[p]
            m.commit(rid, len(tokens) - rc.length)
            live[rid] = tokens
        m.check()
    assert reused > 0


def test_the_pool_is_sized_from_the_free_memory():
    """The arithmetic of `capacity`: by default the pool is what every slot at its full context
    takes, or what fits if that is less; a number that was asked for and does not fit is refused
    with the bytes it needs and the bytes there are; a pool of no page is refused."""
    from hfee_amd.cache import capacity
    from hfee_amd.cache.manager import CacheError
    gib = 1 << 30
    total = 288 * gib
    page = 2 << 20                                     # the 8B shape: 128 KiB a token, 16 tokens
    work = capacity.workspace_bytes(2048, 128256, 28672)
    assert work == 2048 * (4 * 128256 + 16 * 28672)
    reserve = int(capacity.RESERVE_FRACTION * total)
    # plenty of room: the slots' full contexts decide
    assert capacity.choose_pages(None, 8 * 512, 200 * gib, total, work, page) == 8 * 512
    # little room: what fits, to the page
    free = 30 * gib
    fit = (free - work - reserve) // page
    assert capacity.pages_that_fit(free, total, work, page) == fit and 0 < fit < 64 * 8192 // 16
    assert capacity.choose_pages(None, 64 * 8192 // 16, free, total, work, page) == fit
    assert capacity.choose_pages(fit, 1, free, total, work, page) == fit          # asked for: taken as it is
    with pytest.raises(CacheError) as e:
        capacity.choose_pages(fit + 1, 1, free, total, work, page)
    msg = str(e.value)
    assert f"needs {(fit + 1) * page:,} bytes" in msg and f"{free:,}" in msg and f"{fit} pages would fit" in msg
    # the states' bytes come off first
    spare = (free - work - reserve) % page
    assert capacity.pages_that_fit(free, total, work, page, state_bytes=3 * page + spare) == fit - 3
    assert capacity.pages_that_fit(free, total, work, page, state_bytes=3 * page + spare + 1) == fit - 4
    with pytest.raises(CacheError, match="no page of the cache fits"):
        capacity.choose_pages(None, 100, work + reserve + page - 1, total, work, page)
    assert capacity.choose_pages(None, 100, work + reserve + page, total, work, page) == 1


def test_a_chain_of_kept_pages_is_followed_where_it_leads_and_no_further():
    """Prompts that leave a kept chain at each of its pages, or come back to one that another request has lengthened, take
    over what a search by digests alone would, and leave the same digests behind."""
    from hfee_amd.cache.manager import PageDigests

    def digests(tokens, n):
        d = PageDigests(16)
        assert d.cover(tokens, n)
        return list(d.up_to(n))

    base = list(range(100, 100 + 16 * 6 + 5))
    for change in range(0, 16 * 6, 7):
        m = CacheManager([FULL], 16, 64, max_requests=4, keep_prefixes=True)
        for name, tokens in (("a", base), ("b", base[:48] + [7] * 60), ("c", base[:change] + [9] + base[change + 1:])):
            kept = dict(m._kept)
            want = 0
            while want < (len(tokens) - 1) // 16 and digests(tokens, want + 1)[want] in kept:
                want += 1
            rc = m.admit(name, tokens)
            assert rc.length == 16 * want
            m.reserve(name, len(tokens) - rc.length)
            m.commit(name, len(tokens) - rc.length)
            if rc.digests is not None:
                assert rc.digests.cover(tokens, len(tokens) // 16)
                assert rc.digests.up_to(len(tokens) // 16) == digests(tokens, len(tokens) // 16)
            m.release(name, tokens)
            assert set(digests(tokens, len(tokens) // 16)) <= set(m._kept)
            m.check()


def test_outgrown_buffers_of_a_workspace_hold_no_more_than_the_one_in_use():
    """A buffer that grows a little with every step (prompts of ever more rows) leaves those behind that recorded graphs may
    point at: together they stay below it, and it below twice what was asked for."""
    import torch
    from hfee_amd.parts.base import Workspace
    ws = Workspace(8, "cpu")
    kept = []
    for count in range(300, 3000, 7):
        for buf in (ws.flat("product.partial", count, torch.float32), ws.counters("counts", count)):
            assert buf.numel() == count
        kept.append(ws.flat("product.partial", 100, torch.float32).data_ptr())
    for dtype in (torch.float32, torch.int32):
        current, retired = ([b.numel() for b in bufs if b.dtype == dtype] for bufs in (ws._buffers.values(), ws._retired))
        assert len(current) == 1 and current[0] < 2 * 3000 and sum(retired) < current[0]
    assert set(kept) <= {b.data_ptr() for b in [*ws._buffers.values(), *ws._retired]}


@pytest.mark.parametrize("pages,groups,stop", [(1, 1, 1), (5, 1, 0), (5, 2, 3), (40, 3, 40), (40, 1, 39)])
def test_the_native_walks_over_pages(pages, groups, stop):
    """The walks on the manager's own objects against the same in Python: what is left behind, in which order and under what,
    where a chain is left (at its end, at another page's tokens, before its first page), who owns what, and that nothing
    holds on to an object that it has let go."""
    import sys
    from collections import OrderedDict

    from hfee_amd.cache.manager import KEPT, PageDigests
    from hfee_amd.kernels import lib
    native, size, rng = lib.pages(), 128, random.Random(pages + stop)
    tokens = [rng.randrange(1 << 40) for _ in range(16 * pages)]
    own = PageDigests(16)
    assert own.cover(tokens, pages)
    digests, tables = list(own.up_to(pages)), [[1000 * g + 700 + b for b in range(pages)] for g in range(groups)]
    there = digests[pages // 2] if pages > 1 else None
    kept, want = (OrderedDict({there: "kept before"} if there else {}) for _ in range(2))
    behind, stays, twice = None, [], []
    for b in range(pages - 1, -1, -1):
        if digests[b] in want:
            twice.append(b)
        else:
            want[digests[b]] = (tuple(t[b] for t in tables), own.data[b * size:(b + 1) * size], behind)
            stays.append(b)
        behind = digests[b]
    assert native.hfee_keep_pages(kept, digests, tables, own.data, size, pages) == (
        [[t[b] for b in stays] for t in tables], [[t[b] for b in twice] for t in tables])
    assert list(kept.items()) == list(want.items())
    for short in (dict(digests=digests[1:]), dict(data=own.data[1:]), dict(tables=[t[1:] for t in tables])):
        args = dict(dict(digests=digests, tables=tables, data=own.data), **short)
        with pytest.raises(ValueError):
            native.hfee_keep_pages(OrderedDict(), args["digests"], args["tables"], args["data"], size, pages)

    chain = OrderedDict((d, (tuple(t[b] for t in tables), own.data[b * size:(b + 1) * size], digests[b + 1] if b + 1 < pages else None))
                        for b, d in enumerate(digests))
    if stop < pages:                                  # (another page's tokens)
        chain[digests[stop]] = (chain[digests[stop]][0], b"\0" * size, chain[digests[stop]][2])
    refs = [sys.getrefcount(d) for d in digests]
    followed, taken = [], []
    at, after = native.hfee_follow_chain(chain, own.data, size, 0, digests[0], followed, taken)
    assert (at, after) == (stop * size, digests[stop] if stop < pages else None)
    assert followed == digests[:stop] and taken == [tuple(t[b] for t in tables) for b in range(stop)]
    assert list(chain) == digests[stop:]
    del followed, taken, chain, at, after
    assert all(sys.getrefcount(d) <= r for d, r in zip(digests, refs))

    owners = [None] * 4000
    for page in tables[0]:
        owners[page] = "a"
    assert native.hfee_hand_over(owners, tables[0], "a", KEPT) is None and [owners[p] for p in tables[0]] == [KEPT] * pages
    assert native.hfee_hand_over(owners, tables[0], ("kept prefix",), "b") is None           # (equal, not the same)
    owners[tables[0][-1]] = "c"
    assert native.hfee_hand_over(owners, tables[0], "b", "d") == tables[0][-1]
    assert [owners[p] for p in tables[0]] == ["d"] * (pages - 1) + ["c"]
    assert native.hfee_hand_over([None], [0], None, "a") == 0 and native.hfee_hand_over(["a"], [0], "a", None) == 0
    with pytest.raises(IndexError):
        native.hfee_hand_over(owners, [4000], "a", "b")
    with pytest.raises(TypeError):
        native.hfee_hand_over(owners, ["x"], "a", "b")


def test_pages_are_handed_over_by_any_number_that_is_an_index():
    """Page numbers that come out of an array, from a generator, negative ones: as a list's own index takes them; what it refuses is
    refused, and nothing behind it is handed over."""
    import numpy as np
    pool = PagePool(8)
    for _ in range(5):
        pool.take("a")
    pool.hand_over(np.array([0, 1], dtype=np.int32), "a", "b")
    pool.hand_over((p for p in [np.int64(2), -5]), "a", "c")
    pool.hand_over([True], "b", "d")
    assert [pool.owner_of(p) for p in range(6)] == ["b", "d", "c", "c", "a", None]
    for wrong, error in (("x", TypeError), (1.0, TypeError), (8, IndexError), (2 ** 70, IndexError), (5, CacheError)):
        with pytest.raises(error):
            pool.hand_over([wrong, 4], "a", "b")
        assert pool.owner_of(4) == "a"


def test_tokens_as_bytes():
    """Whole numbers of a list as int64; what is no plain one (or no list) is left to the array that takes it; what does not fit is refused."""
    import numpy as np

    from hfee_amd.cache.manager import PageDigests
    from hfee_amd.kernels import lib
    numbers = [0, 1, -1, 128255, 2 ** 63 - 1, -2 ** 63]
    to_bytes = lib.pages().hfee_token_bytes
    assert to_bytes(numbers) == np.asarray(numbers, dtype=np.int64).tobytes() and to_bytes([]) == b""
    assert to_bytes([1, True]) is None and to_bytes([np.int64(3)]) is None and to_bytes((1, 2)) is None
    for wrong in (2 ** 63, -2 ** 63 - 1):
        with pytest.raises(OverflowError):
            to_bytes([1, wrong])
    for tokens in (list(range(16)), np.arange(16), [np.int64(i) for i in range(16)], [True] * 16):
        d = PageDigests(16)
        assert d.cover(tokens, 1) and d.data == np.asarray(tokens, dtype=np.int64).tobytes()


def test_the_walks_library_is_the_hosts_own(tmp_path, monkeypatch):
    """It is compiled and linked without hipcc and needs no HIP runtime; flags that are given are applied, to it too, and make another
    library; and a library is for one layout of Python's objects."""
    import ctypes

    from hfee_amd.kernels import build

    def no_hipcc():
        raise build.BuildError("no hipcc here")
    monkeypatch.setattr(build, "hipcc", no_hipcc)
    monkeypatch.setenv("HFEE_BUILD_DIR", str(tmp_path / "plain"))
    with open(build.build_library("pages"), "rb") as f:
        assert b"libamdhip64" not in f.read()
    plain = build._stamp(*build.library_spec("pages"))
    (tmp_path / "mark.h").write_text('extern "C" __attribute__((visibility("default"))) int hfee_mark() { return 7; }\n')
    monkeypatch.setenv("HFEE_EXTRA_FLAGS", f"-include {tmp_path / 'mark.h'}")
    monkeypatch.setenv("HFEE_BUILD_DIR", str(tmp_path / "marked"))
    assert ctypes.CDLL(build.build_library("pages")).hfee_mark() == 7 and build._stamp(*build.library_spec("pages")) != plain
    monkeypatch.delenv("HFEE_EXTRA_FLAGS")
    monkeypatch.setattr(build, "HOST_FLAGS", [*build.HOST_FLAGS, "-O1"])
    assert build._stamp(*build.library_spec("pages")) != plain
    monkeypatch.undo()
    monkeypatch.setattr(build.sysconfig, "get_config_var", lambda name: "another-abi")
    assert build._stamp(*build.library_spec("pages")) != plain


def test_kept_prefixes_without_the_native_walks(monkeypatch):
    """Where the library cannot be had the manager warns once and does the same in Python: two managers, one each way, through the same
    admissions, steps, releases and pages that run out, agree in everything that they hold; what is refused is refused in both."""
    import warnings

    from hfee_amd.cache import manager, walks
    from hfee_amd.kernels import build, lib

    def unavailable():
        raise lib.KernelLibraryError("no Python.h here")
    with monkeypatch.context() as m:
        m.setattr(lib, "pages", unavailable)
        m.setattr(walks, "_walks", None)
        with pytest.warns(RuntimeWarning, match="no Python.h here"):
            CacheManager([CacheGroupSpec("full", (2, 1, 16), (0,))], 16, 8, 2, keep_prefixes=True)
        with warnings.catch_warnings():
            warnings.simplefilter("error")
            assert walks.walks() is walks.PythonWalks
            CacheManager([CacheGroupSpec("full", (2, 1, 16), (0,))], 16, 8, 2, keep_prefixes=True)
    groups = [CacheGroupSpec("full", (2, 1, 16), (0,)), CacheGroupSpec("full", (2, 2, 16), (1,))]
    both = [CacheManager(groups, 16, 40, 6, keep_prefixes=True) for _ in range(2)]
    sides = (lib.pages(), walks.PythonWalks)
    rng, live, prefix = random.Random(4), {}, [5] * 70
    for step in range(400):
        name, tokens = f"r{step}", None
        if live and (len(live) == 6 or rng.random() < 0.45):
            name = rng.choice(sorted(live))
            tokens, act = live.pop(name), "release"
        else:
            tokens, act = prefix[:rng.randrange(71)] + [rng.randrange(9) for _ in range(rng.randrange(1, 60))], "admit"
            live[name] = tokens
        results = []
        for side, mgr in zip(sides, both):
            with monkeypatch.context() as m:
                m.setattr(manager, "walks", lambda side=side: side)
                if act == "release":
                    mgr.release(name, tokens)
                    results.append(None)
                else:
                    rc = mgr.admit(name, tokens)
                    try:
                        mgr.reserve(name, len(tokens) - rc.length)
                        mgr.commit(name, len(tokens) - rc.length)
                        results.append((rc.length, rc.reused, rc.tables))
                    except OutOfPages:
                        mgr.release(name)
                        results.append("none free")
                mgr.check()
        assert results[0] == results[1]
        if results[0] == "none free":
            del live[name]
        a, b = both
        assert list(a._kept.items()) == list(b._kept.items()) and a.prefix_hits == b.prefix_hits
        assert [(p._free, p._owner) for p in a.pools] == [(p._free, p._owner) for p in b.pools]
    assert both[0].prefix_hits > 1000
    for side in sides:
        with pytest.raises(ValueError):
            side.hfee_keep_pages({}, [b"d"], [[1, 2]], b"\0" * 256, 128, 2)
        with pytest.raises(IndexError):
            side.hfee_hand_over(["a"], [1], "a", "b")
        assert side.hfee_hand_over([None], [0], None, "a") == 0

    monkeypatch.setattr(build, "build_library", lambda name, force=False: unavailable_library() if name == "pages" else name)

    def unavailable_library():
        raise build.BuildError("no Python.h here")
    assert "core" in build.build_all(head_dims=(), kv_sizes=(), mix_sizes=(), kv_sigmoid_sizes=(), mix_vectors_sizes=())
