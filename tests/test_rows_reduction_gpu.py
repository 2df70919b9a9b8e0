"""The reductions behind a Freivalds row at their edges: B of many column chunks and ragged rows,
products of more slices than a wave's lanes, biases under more challenges than one sweep takes,
and fused products of one to many records a row. Against the fp64 oracle."""

from __future__ import annotations

import pytest
import torch

import oracle as O

pytestmark = pytest.mark.gpu
DEV = "cuda"
ROOT = bytes(range(32))

def _product(n, q, w, dtype, bias, seed):
    """Operands on the GPU, P rounded from fp32 sums, one entry off by 64."""
    g = torch.Generator(device=DEV).manual_seed(seed)
    a = torch.randn(n, q, generator=g, device=DEV).to(dtype)
    b = torch.randn(q, w, generator=g, device=DEV).mul_(q ** -0.5).to(dtype)
    bv = torch.randn(w, generator=g, device=DEV).to(dtype).float() if bias else None
    p = a.float() @ b.float()
    if bias:
        p += bv
    p[n // 2, w // 3] += 64.0
    return a, b, p.to(dtype), bv

def _check(row, prod, m, k):
    a, b, p, bv = (None if t is None else t.cpu() for t in prod)
    r = O.challenge_matrices(ROOT, [m], k, p.shape[1])[0]
    want = O.measure_row_f64(a.float(), b.float(), p.float(), r,
                             None if bv is None else bv)
    for c in range(5):  # fp32 sums of non-negative terms
        assert abs(row[c] - want[c]) <= 1e-5 * abs(want[c]), (c, row[c], want[c])
    for j in range(k):  # 64·|r| of the forged entry, or a bf16 product's rounding
        assert abs(row[5 + j] - want[5 + j]) <= 1e-4 * want[5 + j] + 1e-4, (j, row[5 + j], want)

@pytest.mark.parametrize("n,q,w,k,dtype,bias", [
    (70, 45, 9001, 3, torch.bfloat16, False),    # three column chunks of B, ragged everything
    (64, 100, 40000, 4, torch.bfloat16, True),   # ten
    (40000, 33, 20, 2, torch.bfloat16, False),   # 157 slices
    (140000, 16, 5, 1, torch.float32, False),    # 547
    (100, 1000, 17000, 16, torch.float32, True),  # two sweeps of the bias, seventeen chunks
    (33, 5000, 9, 9, torch.float32, True),
    (1, 1, 1, 20, torch.float32, True),
    (257, 31, 33, 255, torch.bfloat16, True),
])
def test_reductions_match_oracle(lib, n, q, w, k, dtype, bias):
    from verification.commitment.native import FvProduct
    prods = [_product(n, q, w, dtype, bias, 3), _product(65, 40, 70, dtype, not bias, 4)]
    plan = lib.fv_plan([FvProduct(a, b, p, m, bv) for m, (a, b, p, bv) in enumerate(prods, 1)], k)
    rows = plan.rows(ROOT).cpu().tolist()
    for m, prod in enumerate(prods, 1):
        _check(rows[m - 1], prod, m, k)
    plan.close()

@pytest.mark.parametrize("k", [1, 2, 4])
@pytest.mark.parametrize("dtype,n,w", [
    (torch.bfloat16, 64, 512), (torch.bfloat16, 193, 2048), (torch.bfloat16, 65, 8192),
    (torch.bfloat16, 64, 16384 + 512), (torch.float32, 127, 1024)])
def test_fused_records_match_oracle(lib, dtype, n, w, k):
    """2 to 34 records a row; the second product's rows begin inside a block of 64."""
    from verification.commitment import native
    prods = [_product(n, 48, w, dtype, False, 5), _product(128, 40, w, dtype, False, 6)]
    fv = lib.fv_plan([native.FvProduct(a, b, p, m, bv)
                      for m, (a, b, p, bv) in enumerate(prods, 1)], k)
    ps = [prod[2] for prod in prods]
    leaf = lib.leaf_plan([O.tensor_leaf_header(3, p) for p in ps], ps,
                         [native.FINITE_KIND[dtype]] * 2, fuse=fv)
    assert leaf.fused >= 1
    key = torch.tensor(list(ROOT), dtype=torch.uint8, device=DEV)
    digests = torch.empty(2, 32, dtype=torch.uint8, device=DEV)
    bad = torch.empty(1, dtype=torch.int32, device=DEV)
    rows = torch.empty(2, 5 + k, dtype=torch.float64, device=DEV)
    lib.step_run(leaf, fv, key, digests, bad, rows)
    for m, prod in enumerate(prods, 1):
        _check(rows.cpu().tolist()[m - 1], prod, m, k)
    assert [bytes(x) for x in digests.cpu().numpy()] == \
        [O.tensor_leaf_hash(3, p.cpu()) for p in ps]
    fv.close()

@pytest.mark.parametrize("k", [1, 4, 64, 255])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_wide_products_under_few_and_many_challenges(lib, dtype, k):
    """Small plans whose chunks are cut as far as their columns and challenges say: a wide A, a
    wide B and P."""
    from verification.commitment.native import FvProduct
    prods = [_product(40, 9001, 70, dtype, False, 7), _product(70, 45, 9001, dtype, True, 8)]
    plan = lib.fv_plan([FvProduct(a, b, p, m, bv) for m, (a, b, p, bv) in enumerate(prods, 1)], k)
    rows = plan.rows(ROOT).cpu().tolist()
    for m, prod in enumerate(prods, 1):
        _check(rows[m - 1], prod, m, k)
    plan.close()

@pytest.mark.parametrize("k", [1, 2, 4])
def test_fused_rows_short_and_long_match_oracle(lib, k):
    """A plan of rows of few and of many records, either side of the line between them (48 slots),
    whose products are not in that order."""
    from verification.commitment import native
    # (rows in whole waves of a period, so that no class is padded and all are fused,
    # but the last, whose rows fit no period); the two widest have chunks enough to be added up ahead
    # of the rows, unless they are fused
    shapes = [(64, 24576), (64, 512), (64, 24064), (192, 2048), (64, 65536), (320, 1024), (33, 65537)]
    prods = [_product(n, 16, w, torch.bfloat16, False, 20 + i) for i, (n, w) in enumerate(shapes)]
    fv = lib.fv_plan([native.FvProduct(a, b, p, m, bv)
                      for m, (a, b, p, bv) in enumerate(prods, 1)], k)
    ps = [prod[2] for prod in prods]
    leaf = lib.leaf_plan([O.tensor_leaf_header(3, p) for p in ps], ps,
                         [native.KIND_BF16] * len(ps), fuse=fv)
    assert leaf.fused == 6
    key = torch.tensor(list(ROOT), dtype=torch.uint8, device=DEV)
    digests = torch.empty(len(ps), 32, dtype=torch.uint8, device=DEV)
    bad = torch.empty(1, dtype=torch.int32, device=DEV)
    rows = torch.empty(len(ps), 5 + k, dtype=torch.float64, device=DEV)
    lib.step_run(leaf, fv, key, digests, bad, rows)
    for m, prod in enumerate(prods, 1):
        _check(rows.cpu().tolist()[m - 1], prod, m, k)
    fv.close()

@pytest.mark.parametrize("k", [1, 2, 3, 4])
def test_reductions_of_a_few_rows(lib, k):
    """B of every height around the rows a block reduces at each k (128, 64, 64, 32), side by side."""
    from verification.commitment.native import FvProduct
    heights = (1, 31, 32, 33, 63, 64, 65, 96, 97, 127, 128, 129, 160, 257)
    prods = [_product(9, q, 40, torch.float32, i % 3 == 0, 30 + i) for i, q in enumerate(heights)]
    prods += [_product(9, q, 5000, torch.bfloat16, False, 50 + q) for q in (33, 65, 129)]
    plan = lib.fv_plan([FvProduct(a, b, p, m, bv) for m, (a, b, p, bv) in enumerate(prods, 1)], k)
    rows = plan.rows(ROOT).cpu().tolist()
    for m, prod in enumerate(prods, 1):
        _check(rows[m - 1], prod, m, k)
    plan.close()
