"""Staged leaves (messages not word aligned where they lie): every header length and payload
alignment, from device and host memory, beside leaves hashed in place. Bit for bit against the
CPU oracle. And a root set from host memory."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle as O

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("host", [False, True])
def test_headers_and_alignments(lib, host):
    g = torch.Generator().manual_seed(5)
    store = torch.randint(0, 256, (80_000,), generator=g, dtype=torch.uint8)
    src = store if host else store.to(DEV)
    heads, spans = [], []
    for i, n in enumerate((0, 1, 2, 3, 4, 5, 15, 16, 17, 31, 32, 33, 1000, 1023, 1024, 1025, 4075,
                           4096, 4097, 9000, 16385, 40001)):
        for hl in (0, 1, 2, 3, 5, 15, 16, 21):
            heads.append(bytes((i + j) & 255 for j in range(hl)))
            spans.append((3 * i + hl, n))
    n = len(heads)
    hdr_len = np.array([len(h) for h in heads], np.uint32)
    hdr_off = np.concatenate([[0], np.cumsum(hdr_len[:-1])]).astype(np.uint64)
    ptr = np.array([src.data_ptr() + o for o, _ in spans], np.uint64)
    ln = np.array([k for _, k in spans], np.uint64)
    raw = store.numpy().tobytes()
    want = [O.hash_leaf(h, raw[o:o + k]) for h, (o, k) in zip(heads, spans)]
    d, bad = lib.hash_leaves(b"".join(heads), hdr_off, hdr_len, np.arange(n, dtype=np.uint32), ptr,
                             ln, np.zeros(n, np.uint8))
    assert bad == n and [bytes(x) for x in d] == want


def test_root_from_host_memory(lib):
    key = torch.empty(3, 32, dtype=torch.uint8, device=DEV)
    roots = [bytes((7 * i + j) & 255 for j in range(32)) for i in range(3)]
    for i, r in enumerate(roots):
        lib.set_key(key[i], r)
    assert [bytes(x) for x in key.cpu().numpy()] == roots
    for bad in (roots[0][:31], roots[0] + b"x"):
        with pytest.raises(ValueError):
            lib.set_key(key[0], bad)
    with pytest.raises(ValueError):
        lib.set_key(key, roots[0])


def test_rows_under_a_host_root_or_a_device_one(lib):
    from verification.commitment.native import FvProduct
    a, b = torch.randn(40, 33, device=DEV), torch.randn(33, 50, device=DEV)
    x, y = a.bfloat16(), b.bfloat16()
    plan = lib.fv_plan([FvProduct(a, b, a @ b, 1), FvProduct(x, y, x @ y, 2)], 3)
    root = bytes(range(100, 132))
    store = torch.zeros(40, dtype=torch.uint8, device=DEV)
    want = plan.rows(root)
    for skip in (0, 1, 4):  # a device root at any alignment
        store[skip:skip + 32] = torch.tensor(list(root), dtype=torch.uint8)
        assert torch.equal(plan.rows(store[skip:skip + 32]), want)
    with pytest.raises(ValueError):
        plan.rows(root[:31])
    plan.close()
