"""Row passes over operands at any alignment (views at odd offsets, odd row strides) and widths
around the edges of K-steps, stages and chunks, both where a block shares V and where each lane
loads its own (a limited grid). Against the fp64 oracle."""

from __future__ import annotations

import pytest
import torch

import oracle as O

pytestmark = pytest.mark.gpu
DEV = "cuda"
ROOT = bytes(range(32))
WIDTHS = (1, 7, 8, 9, 15, 16, 17, 31, 32, 33, 63, 64, 65, 127, 128, 129, 160, 255, 257, 391)


def _view(t, skip, pad):
    """``t`` as a view `skip` elements into its storage whose rows are `pad` elements apart, with
    NaN in every element between them: a load that used one would show."""
    rows, cols = t.shape
    flat = torch.full((skip + rows * (cols + pad),), float("nan"), dtype=t.dtype, device=DEV)
    out = flat[skip:].view(rows, cols + pad)[:, :cols]
    return out.copy_(t)


@pytest.mark.parametrize("k", [1, 4, 16, 40])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_any_alignment(lib, dtype, k):
    from verification.commitment.native import FvProduct
    prods = []
    for i, q in enumerate(WIDTHS):
        n, w = 17 + 5 * i, WIDTHS[-1 - i]
        g = torch.Generator(device=DEV).manual_seed(i)
        a = torch.randn(n, q, generator=g, device=DEV).to(dtype)
        b = torch.randn(q, w, generator=g, device=DEV).mul_(q ** -0.5).to(dtype)
        p = a.float() @ b.float()
        p[n // 2, w // 2] += 64.0
        prods.append((_view(a, i % 9, i % 4), _view(b, (i + 3) % 7, i % 3),
                      _view(p.to(dtype), (i + 1) % 5, (i + 1) % 4)))
    # a chunk's end inside a K-step, in a matrix of several chunks
    wide = 8 * 1024 + 13
    a = torch.randn(40, wide, device=DEV).to(dtype)
    b = torch.randn(wide, 50, device=DEV).mul_(wide ** -0.5).to(dtype)
    p = a.float() @ b.float()
    p[3, 4] += 64.0
    prods.append((_view(a, 1, 2), _view(b, 3, 0), _view(p.to(dtype), 0, 1)))
    plan = lib.fv_plan([FvProduct(*x, m) for m, x in enumerate(prods, 1)], k)
    rows = plan.rows(ROOT).cpu()
    for m, (a, b, p) in enumerate(prods, 1):
        a, b, p = a.cpu().float(), b.cpu().float(), p.cpu().float()
        r = O.challenge_matrices(ROOT, [m], k, p.shape[1])[0]
        want = O.measure_row_f64(a, b, p, r)
        got = rows[m - 1].tolist()
        for c in range(5):
            assert abs(got[c] - want[c]) <= 1e-5 * abs(want[c]), (m, c, got[c], want[c])
        for j in range(5, 5 + k):
            assert abs(got[j] - want[j]) <= 1e-4 * want[j] + 1e-4, (m, j, got[j], want[j])
    for stage in (1, 3, 4):
        plan.set_grid(stage, 3)
    assert torch.equal(plan.rows(ROOT).cpu(), rows)
    plan.close()
