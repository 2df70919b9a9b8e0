"""``pots_hash_leaves`` where its calls share memory: results and metadata beyond the 1 MiB pinned
regions, and several threads at once. Bit for bit against the CPU oracle."""

from __future__ import annotations

import threading

import numpy as np
import pytest
import torch

import oracle as O

pytestmark = pytest.mark.gpu


def _messages(n, seed):
    """``n`` messages that are headers alone, 0 to 40 bytes: ``hash_leaves``' arguments and the
    digests."""
    rng = np.random.default_rng(seed)
    lens = rng.integers(0, 41, n).astype(np.uint32)
    buf = rng.integers(0, 256, int(lens.sum()) + 1, dtype=np.uint8).tobytes()
    offs = np.concatenate([[0], np.cumsum(lens[:-1], dtype=np.uint64)]).astype(np.uint64)
    zero = np.zeros(n, np.uint64)
    args = (buf, offs, lens, np.arange(n, dtype=np.uint32), zero, zero, np.zeros(n, np.uint8))
    want, bad = O.hash_leaves([(buf[int(o):int(o) + int(l)], b"", 0)
                               for o, l in zip(offs, lens)])
    assert bad == n
    return args, want


@pytest.mark.parametrize("n", [5000, 32767, 32768, 40000])
def test_past_the_pinned_regions(lib, n):
    """5000 leaves' metadata and 32768 leaves' digests are just past 1 MiB."""
    args, want = _messages(n, n)
    for _ in range(2):
        d, bad = lib.hash_leaves(*args)
        assert bad == n and [bytes(x) for x in d] == want


def test_threads_at_once(lib):
    cases = [_messages(n, 7 + i) for i, n in enumerate((1, 300, 5000, 33000))]
    wrong, start = [], threading.Barrier(len(cases))

    def work(args, want):
        start.wait()
        for _ in range(12):
            d, bad = lib.hash_leaves(*args)
            if bad != len(want) or [bytes(x) for x in d] != want:
                wrong.append(len(want))

    threads = [threading.Thread(target=work, args=case) for case in cases]
    for t in threads:
        t.start()
    for t in threads:
        t.join(90)
    assert not any(t.is_alive() for t in threads) and wrong == []
