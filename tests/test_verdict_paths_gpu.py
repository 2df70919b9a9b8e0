"""Verdicts on either side of the rule that picks one block for all products or a thread each, by
products and challenges: codes and the smallest rejected index equal the oracle's."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle as O

pytestmark = pytest.mark.gpu
BF16, FP32 = 2.0**-8, 2.0**-24


@pytest.mark.parametrize("n, k", [(1, 255), (256, 33), (257, 31), (257, 32), (1024, 8), (1024, 9),
                                  (1025, 1), (700, 40)])
def test_codes_and_first_rejection(lib, n, k):
    from verification.commitment import native
    rng = np.random.default_rng(n + k)
    rows = np.concatenate([rng.lognormal(0, 0.1, (n, 4)), np.zeros((n, 1)),
                           rng.lognormal(-12, 1, (n, k))], axis=1)
    for i in {n - 1, n // 2, min(n - 1, 255)}:  # a residual over its band, a late challenge's
        rows[i, 5 + k - 1 - i % min(k, 3)] = 1e3
    rows[n // 3, 2] = np.nan
    specs = native.verdict_specs([64] * n, [100] * n, [False] * n, [1e4] * n)
    want = [O.judge(O.finish_row(r.tolist(), q=64, n=100, eps_in=BF16, eps_acc=FP32, biased=False),
                    tau=8.0, kappa_max=1e4) for r in rows]
    for r, w in ((rows, want), (rows[::-1].copy(), want[::-1])):
        codes, _, first = lib.verdicts(torch.from_numpy(r).cuda(), specs, k=k, eps_in=BF16,
                                       eps_acc=FP32, tau=8.0)
        assert [tuple(c) for c in codes.cpu().tolist()] == w
        assert int(first) == min(i for i, c in enumerate(w) if c[0] != 0)
