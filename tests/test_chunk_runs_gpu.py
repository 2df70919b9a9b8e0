"""A lane's run of consecutive chunks, at each length (a plan by itself takes four only from 16 Mi
chunks on): the carry from one chunk to the next, runs that end a leaf early, and the fused
leaves' runs over classes and periods. Digests bit for bit against the CPU oracle; a fused plan's
rows against the unfused plan's, relative 1e-6 as the fused plan's tests hold them."""

from __future__ import annotations

import pytest
import torch

import oracle as O
from test_fused_gpu import KEY, _product
from test_hash_paths_gpu import DEV, _leaves, _values

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("run", [1, 2, 3, 4])
def test_plain_runs_match_oracle(lib, run):
    from verification.commitment import native
    ts = _leaves()
    for i, chunks in enumerate((2, 3, 4, 5, 6, 7, 8, 9, 12, 13, 31)):
        for j, tail in enumerate((0, 4, 64, 124, 128, 1000)):  # the last chunk's bytes, 0: all
            nbytes = 1024 * (chunks - (tail > 0)) + tail - 8
            flat = _values(nbytes // 4 + 3, torch.float32, 40 * i + j).to(DEV)
            ts.append(flat[j % 4:j % 4 + nbytes // 4])  # payloads at every word shift
    want, bad = O.hash_leaves([(O.tensor_leaf_header(3, t), t.cpu(), O.FINITE_KIND[t.dtype])
                               for t in ts], simd=O.simd_degree() > 1)
    assert bad == len(ts)
    plan = lib.leaf_plan([O.tensor_leaf_header(3, t) for t in ts], ts,
                         [native.FINITE_KIND[t.dtype] for t in ts], run=run)
    for grid in (0, 2):
        plan.set_grid(grid)
        d, first_bad = plan.run()
        assert int(first_bad) == len(ts)
        assert [bytes(x) for x in d.cpu().numpy()] == want
    for at in (-1, 4 * 256 + 3, 255, 0):  # a value of the last leaf's last, fifth, first chunk
        ts[-1][at] = float("inf")
        assert int(plan.run()[1]) == len(ts) - 1
        ts[-1][at] = 1.0
    plan.close()
    with pytest.raises(ValueError):
        lib.leaf_plan([O.tensor_leaf_header(3, ts[0])], ts[:1], [0], run=5)


# rows (bytes / 1024 = classes per period): one class in several periods, rounded up and exact, two,
# three, as many as a run, more with a ragged last range, many; few periods (runs of one instead)
SHAPES = [(torch.bfloat16, 1000, 512), (torch.bfloat16, 950, 512), (torch.bfloat16, 512, 1024),
          (torch.bfloat16, 64, 1536), (torch.bfloat16, 64, 2048), (torch.bfloat16, 127, 2560),
          (torch.bfloat16, 64, 3584), (torch.bfloat16, 4090, 520), (torch.float32, 255, 1024),
          (torch.float32, 4090, 260)]


@pytest.mark.parametrize("k", [1, 4])
@pytest.mark.parametrize("run", [1, 2, 3, 4])
def test_fused_runs_match_unfused(lib, run, k):
    from verification.commitment import native
    for dtype in (torch.bfloat16, torch.float32):
        prods = [[t.to(DEV) for t in _product(n, 48, w, dt, 3 + i)]
                 for i, (dt, n, w) in enumerate(SHAPES) if dt == dtype]
        ps = [p for _, _, p in prods]
        heads = [O.tensor_leaf_header(O.TAG_PRODUCT, p) for p in ps]
        kinds = [native.FINITE_KIND[dtype]] * len(ps)
        key = torch.tensor(list(KEY), dtype=torch.uint8, device=DEV)
        fvp = [native.FvProduct(a, b, p, m) for m, (a, b, p) in enumerate(prods, 1)]
        plain = lib.fv_plan(fvp, k)
        rows_u = plain.rows(key).cpu()
        fv = lib.fv_plan(fvp, k)
        leaf = lib.leaf_plan(heads, ps, kinds, fuse=fv, run=run)
        assert leaf.fused == len(ps)
        dig = torch.empty(len(ps), 32, dtype=torch.uint8, device=DEV)
        bad = torch.empty(1, dtype=torch.int32, device=DEV)
        rows = torch.empty(len(ps), 5 + k, dtype=torch.float64, device=DEV)
        for _ in range(2):
            lib.step_run(leaf, fv, key, dig, bad, rows)
            assert int(bad) == len(ps)
            assert [bytes(x) for x in dig.cpu().numpy()] == \
                [O.tensor_leaf_hash(O.TAG_PRODUCT, p.cpu()) for p in ps]
            assert torch.allclose(rows.cpu()[:, :5], rows_u[:, :5], rtol=1e-6, atol=0)
        fv.close()
        plain.close()
