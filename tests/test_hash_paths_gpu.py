"""The leaf hasher's ways of cutting work, each against the CPU oracle bit for bit: chunks on
four lanes and one lane per chunk, chosen by a plan's chunk count (runs of chunks per lane take
16 GiB of leaves: the full-size configurations' tests)."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle as O

pytestmark = pytest.mark.gpu
DEV = "cuda"
KINDS = (torch.float32, torch.bfloat16, torch.float16, torch.int32)


def _values(n, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    if dtype == torch.int32:
        return torch.randint(-2**31, 2**31 - 1, (n,), generator=g, dtype=torch.int32)
    return torch.randn(n, generator=g).to(dtype)


def _leaves():
    """Lengths around the edges of words, 16-byte groups, blocks, pairs of blocks and chunks
    (the header takes the first 8, 12 or 16 bytes of a message), from payloads at every word
    shift, as 1-D to 3-D tensors."""
    out = []
    for i, nbytes in enumerate((4, 8, 12, 16, 20, 44, 48, 52, 56, 60, 64, 108, 112, 116, 120, 128,
                                1000, 1004, 1008, 1012, 1016, 1020, 1024, 1028, 2036, 2040, 2044,
                                4084, 4088, 5000, 16 * 1024 - 12, 16 * 1024 - 8, 70000)):
        dtype = KINDS[i % 4]
        n = nbytes // dtype.itemsize
        pad = (i % 5) * (4 // min(4, dtype.itemsize))  # 4-byte steps: word shifts of the payload
        flat = _values(n + pad, dtype, 100 + i).to(DEV)[pad:]
        out.append(flat.view([(n,), (1, n), (1, n, 1)][i % 3]))
    odd = _values(3001, torch.bfloat16, 7).to(DEV)
    return out + [odd[1:2], odd[1:], odd[3:2000]]  # 2-byte aligned: staged


@pytest.mark.parametrize("filler_mib", [0, 33, 513])  # quads; a chunk per lane, few and many
def test_chunk_paths_match_oracle(lib, filler_mib):
    from verification.commitment import native
    ts = _leaves()
    if filler_mib:
        ts.append(torch.randn(filler_mib * 262144 - 5, device=DEV))
    want, bad = O.hash_leaves([(O.tensor_leaf_header(3, t), t.cpu(), O.FINITE_KIND[t.dtype])
                               for t in ts], simd=O.simd_degree() > 1)
    assert bad == len(ts)
    plan = lib.leaf_plan([O.tensor_leaf_header(3, t) for t in ts], ts,
                         [native.FINITE_KIND[t.dtype] for t in ts])
    d, first_bad = plan.run()
    assert int(first_bad) == len(ts)
    assert [bytes(x) for x in d.cpu().numpy()] == want
    # a NaN in a leaf's last value, then in the first value of an earlier one
    floats = [i for i, t in enumerate(ts[:33]) if t.dtype != torch.int32]
    for i, at in ((floats[-1], -1), (floats[3], 0)):
        ts[i].view(-1)[at] = float("nan")
        assert int(plan.run()[1]) == i
    plan.set_grid(3)  # a block limit: the same digests
    for i in floats:
        ts[i].view(-1)[0 if i == floats[3] else -1] = 1.0
    a = plan.run()[0].cpu()
    plan.set_grid(0)
    assert torch.equal(a, plan.run()[0].cpu())
    plan.close()


def test_messages_with_no_payload(lib):
    """Host messages are headers alone: every length around a block and a chunk."""
    msgs = [bytes((7 * i + j) & 255 for j in range(n)) for i, n in enumerate(
        (0, 1, 2, 3, 4, 15, 16, 17, 62, 63, 64, 65, 127, 128, 1022, 1023, 1024, 1025, 3071))]
    n = len(msgs)
    lens = np.array([len(m) for m in msgs], np.uint32)
    offs = np.concatenate([[0], np.cumsum(lens[:-1])]).astype(np.uint64)
    zero = np.zeros(n, np.uint64)
    d, bad = lib.hash_leaves(b"".join(msgs), offs, lens, np.arange(n, dtype=np.uint32), zero, zero,
                             np.zeros(n, np.uint8))
    assert bad == n
    assert [bytes(x) for x in d] == [O.hash_leaf(m) for m in msgs]


@pytest.mark.parametrize("chunks", [
    [2, 127, 128, 129, 130, 255, 257, 1022, 1023, 1024, 1025, 1026, 1151, 1152, 1153, 2047, 2048,
     2049, 3000],            # a tile's quads alone, its wide levels, one tile and several
    [1024 * 1024 + 1],       # three folds, the last tile a single node promoted through two
    [1024 * 1024, 1024 * 1025 - 1]])
def test_leaf_trees_at_tile_edges(lib, chunks):
    from verification.commitment import native
    ts = [torch.randint(0, 2**31 - 1, ((1024 * n - 100) // 4,), device=DEV, dtype=torch.int32)
          for n in chunks]
    heads = [O.tensor_leaf_header(2, t) for t in ts]
    want, _ = O.hash_leaves([(h, t.cpu(), 0) for h, t in zip(heads, ts)],
                            simd=O.simd_degree() > 1)
    plan = lib.leaf_plan(heads, ts, [native.KIND_NONE] * len(ts))
    assert plan.chunks == sum(chunks)
    assert [bytes(x) for x in plan.run()[0].cpu().numpy()] == want
    plan.close()


@pytest.mark.parametrize("n", [1, 2, 3, 127, 128, 129, 255, 256, 257, 258, 511, 512, 513, 65535,
                               65536, 65537, 65793, 100003])
def test_outer_tree_at_tile_edges(lib, n):
    d = torch.randint(0, 256, (n, 32), device=DEV, dtype=torch.uint8)
    want = O.merkle_tree([bytes(x) for x in d.cpu().numpy()])
    assert lib.merkle_tree_device(d).cpu().numpy().tobytes() == want


@pytest.mark.parametrize("short", [7999, 8000])  # a block a leaf, a lane per eight nodes
def test_leaf_trees_of_many_short_leaves(lib, short):
    """Short leaves of every shape around a lane's eight nodes and its folds, up to 512 chunks, and
    longer ones and single chunks among them."""
    from verification.commitment import native
    edges = [2, 3, 7, 8, 9, 10, 15, 16, 17, 63, 64, 65, 72, 73, 511, 512]
    chunks = edges + [2 + i % 9 for i in range(short - len(edges))]
    for at, c in ((0, 513), (7, 1), (100, 1025), (len(chunks) // 2, 2049), (len(chunks), 1)):
        chunks.insert(at, c)
    flat = torch.randint(0, 2**31 - 1, (sum(chunks) * 256,), device=DEV, dtype=torch.int32)
    ts, at = [], 0
    for i, c in enumerate(chunks):
        n = (1024 * c - 8 - 4 * (i % 200)) // 4
        ts.append(flat[at:at + n])
        at += n
    heads = [O.tensor_leaf_header(2, t) for t in ts]
    host, at, items = flat.cpu(), 0, []
    for h, t in zip(heads, ts):
        items.append((h, host[at:at + t.numel()], 0))
        at += t.numel()
    want, _ = O.hash_leaves(items, simd=O.simd_degree() > 1)
    plan = lib.leaf_plan(heads, ts, [native.KIND_NONE] * len(ts))
    assert plan.chunks == sum(chunks)
    for _ in range(2):
        assert [bytes(x) for x in plan.run()[0].cpu().numpy()] == want
    plan.close()


@pytest.mark.parametrize("step", [256, 257])  # words between payloads: one word shift, all four
@pytest.mark.parametrize("kind", ["none", "float"])
def test_runs_of_many_short_leaves(lib, step, kind):
    """Leaves of 2 to 5 chunks and around the lengths that take runs of four, past the number from
    which they do; longer ones and single chunks among them."""
    from verification.commitment import native
    edges = [5, 6, 7, 8, 9, 12, 15, 16, 18, 19, 20, 23, 24, 25, 27, 28, 64, 127, 128, 129, 132]
    chunks = [2 + i % 3 for i in range(65400)] + edges * 8 + [1, 500, 2048]
    tails = (0, 1, 16, 17, 31, 32, 33, 250)  # words the last chunk lacks
    flat = torch.randn(1 << 20, device=DEV)
    host = flat.cpu()
    ts, items, at = [], [], 0
    for i, c in enumerate(chunks):
        n = 256 * c - 2 - tails[i % len(tails)]
        at = (at + step) % ((1 << 20) - 256 * 2049)
        ts.append(flat[at:at + n])
        items.append((at, n))
    k = native.KIND_NONE if kind == "none" else native.KIND_F32
    heads = [O.tensor_leaf_header(2, t) for t in ts]
    want, _ = O.hash_leaves([(h, host[a:a + n], 0) for h, (a, n) in zip(heads, items)],
                            simd=O.simd_degree() > 1)
    plan = lib.leaf_plan(heads, ts, [k] * len(ts))
    d, bad = plan.run()
    assert int(bad) == len(ts) and [bytes(x) for x in d.cpu().numpy()] == want
    if kind == "float":  # the second chunk's first word and the last word of one leaf
        for word in (items[70][0] + 254, items[70][0] + items[70][1] - 1):
            flat[word] = float("nan")
            first = next(i for i, (a, n) in enumerate(items) if a <= word < a + n)
            assert int(plan.run()[1]) == first
            flat[word] = 1.0
    plan.close()
