"""The walks over the pages of kept prefixes on the manager's own objects: native (csrc/pages.cpp) where that library can be had,
the same here in Python where it cannot (no C++ compiler, no headers of this Python): the manager is bookkeeping and runs
without either, only slower (admitting and releasing 64 requests of 385 tokens 3.3 ms instead of 2.2).
"""
from __future__ import annotations

import warnings

from ..kernels import lib


class PythonWalks:
    @staticmethod
    def hfee_token_bytes(tokens):
        """The numbers as int64, one after the other, in bytes, or None for "by way of an array"."""
        return None

    @staticmethod
    def hfee_follow_chain(kept, data, page_bytes, at, following, digests, taken):
        """Follows a chain of kept pages (digest -> (pages, the page's tokens as bytes, the digest of the page behind it)): from byte
        `at` of data on, as long as the entry under `following` holds the next page's bytes, it leaves `kept`, its digest
        is added to `digests` and its pages to `taken`.  Returns (the byte that it came to, the digest that is followed there)."""
        while following is not None and at + page_bytes <= len(data):
            entry = kept.get(following)
            if entry is None or entry[1] != data[at:at + page_bytes]:
                break
            del kept[following]
            digests.append(following)
            taken.append(entry[0])
            at, following = at + page_bytes, entry[2]
        return at, following

    @staticmethod
    def hfee_keep_pages(kept, digests, tables, data, page_bytes, n):
        """Leaves the first `n` pages of a request (`tables`: a list of pages a group) behind in `kept`, the deepest first.  Returns
        (the pages of those that stay, the pages of those that were kept already), a list a group each."""
        if min(len(digests), len(data) // page_bytes, *(len(t) for t in tables)) < n:
            raise ValueError("keep_pages: fewer digests, pages or tokens than pages to keep")
        stays, twice, behind = [[] for _ in tables], [[] for _ in tables], None
        for b in range(n - 1, -1, -1):
            there = digests[b] in kept
            if not there:
                kept[digests[b]] = (tuple(t[b] for t in tables), data[b * page_bytes:(b + 1) * page_bytes], behind)
            for pages, table in zip(twice if there else stays, tables):
                pages.append(table[b])
            behind = digests[b]
        return stays, twice

    @staticmethod
    def hfee_hand_over(owners, pages, owner, new_owner):
        """owners[page] <- new_owner for every page, as long as it is `owner`'s.  Returns None, or the first page that is not."""
        for page in pages:
            if owners[page] != owner or owner is None or new_owner is None:
                return page
            owners[page] = new_owner
        return None


_walks = None


def walks():
    """The native walks, or those in Python; which one is settled by the first call."""
    global _walks
    if _walks is None:
        try:
            _walks = lib.pages()
        except lib.KernelLibraryError as e:
            warnings.warn(f"the walks over kept pages are in Python, which is slower: {e}", RuntimeWarning, stacklevel=2)
            _walks = PythonWalks
    return _walks
