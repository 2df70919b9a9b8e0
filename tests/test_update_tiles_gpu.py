"""Check 6a's kernel at the edges of its blocks and steps, and where an entry is decided without
a division: bands at an entry's own ratio and a bit to either side, ties, zero and non-finite
values, bands of zero and below. Bit for bit against the CPU oracle."""

from __future__ import annotations

import math

import pytest
import torch

import oracle as O

pytestmark = pytest.mark.gpu
DEV = "cuda"
EPS_W, ETA = 2.0**-24, 1e-3


def _case(n, seed, dtypes):
    g = torch.Generator().manual_seed(seed)
    w = torch.randn(n, generator=g)
    parts = [torch.randn(n, generator=g).to(dt) for dt in dtypes]
    grad = O.chain_gradient(parts)
    wn = torch.add(w, grad, alpha=-ETA)
    # a few entries off by several ulps, one pair of them tied
    for i in torch.randint(0, n, (5,), generator=g).tolist():
        for _ in range(i % 4):
            wn[i] = torch.nextafter(wn[i], torch.tensor(math.inf))
    return w, wn, parts


def _check(lib, cases, skip=0):
    from verification.commitment import native

    def put(t):  # `skip` elements into an allocation: not 16-byte aligned when it is 1
        flat = torch.empty(t.numel() + skip, dtype=t.dtype, device=DEV)[skip:]
        return flat.copy_(t)

    plan = lib.update_plan([native.UpdateWeight(put(w), put(wn), [put(p) for p in parts], tau)
                            for w, wn, parts, tau in cases], ETA, EPS_W)
    got = native.UpdatePlan.decode(plan.run())
    plan.close()
    for (w, wn, parts, tau), (rho, nf, over) in zip(cases, got):
        want = O.update_identity(w, wn, parts, ETA, EPS_W, tau)
        assert (rho == want["rho_max"] or math.isnan(rho) and math.isnan(want["rho_max"])), \
            (len(w), tau, rho, want)
        assert (nf, over) == (want["first_nonfinite"], want["first_over"]), (len(w), tau, want)


@pytest.mark.parametrize("skip", [0, 1])
@pytest.mark.parametrize("dtypes", [[torch.bfloat16], [torch.float32, torch.bfloat16],
                                    [torch.bfloat16] * 3])
def test_sizes_and_bands(lib, dtypes, skip):
    cases = []
    for i, n in enumerate((1, 3, 4, 255, 1023, 4095, 4096, 4097, 16383, 16384, 16385, 40001)):
        w, wn, parts = _case(n, i, dtypes)
        top = O.update_identity(w, wn, parts, ETA, EPS_W, 4.0)["rho_max"]
        for tau in (4.0, top, math.nextafter(top, 0.0), math.nextafter(top, math.inf), 0.0):
            cases.append((w, wn, parts, tau))
    _check(lib, cases, skip)
    for n in ((1 << 20) + 3, (8 << 20) + 3):  # with these, the plan's wider blocks
        w, wn, parts = _case(n, 77, dtypes)
        _check(lib, [*cases, (w, wn, parts, 4.0)], skip)


INF, NAN, BIG, TINY = math.inf, math.nan, 3.4e38, 1e-45
# (entry, its W_t, W_{t+1} and gradient)
SPECIAL = [(5, 0.0, 0.0, 0.0), (5, 0.0, 1.0, 0.0), (5, 0.0, TINY, 0.0), (5, 1.0, INF, 0.0),
           (5, INF, 1.0, 0.0), (5, INF, INF, 0.0), (5, NAN, 1.0, 0.0), (5, 1.0, NAN, 0.0),
           (5, 1.0, 1.0, NAN), (5, 1.0, 1.0, INF), (5, BIG, -BIG, 0.0), (5, TINY, -TINY, 0.0),
           (4100, 0.0, 1.0, 0.0), (4100, NAN, NAN, NAN), (20000, 1.0, 2.0, 1.0)]


def _special(taus):
    cases = []
    for seed, (at, w_v, wn_v, g_v) in enumerate(SPECIAL):
        w, wn, parts = _case(20001, 50 + seed, [torch.float32])
        w[at], wn[at], parts[0][at] = w_v, wn_v, g_v
        cases += [(w, wn, parts, tau) for tau in taus]
    return cases


def test_special_values(lib):
    cases = _special((4.0, 1e30, 0.0))
    zero = torch.zeros(300)
    cases += [(zero, zero, [zero], tau) for tau in (4.0, 0.0, -1.0, math.nan)]
    w, wn, parts = _case(300, 99, [torch.float32])
    cases += [(w, wn, parts, tau) for tau in (-1.0, math.nan, math.inf, 5e-324)]
    _check(lib, cases)
    for n in (1 << 20, 8 << 20):  # with these, the plan's wider blocks
        w, wn, parts = _case(n, 78, [torch.float32])
        _check(lib, [*cases, (w, wn, parts, 4.0)])


@pytest.mark.parametrize("tau", [math.inf, 1e308, 1e300, 1e270, -math.inf])
def test_special_values_under_bands_past_fp64s_products(lib, tau):
    """tau·scale overflows fp64 (or, at 1e270, nearly): an infinite residual lies within it."""
    cases = _special((tau,))
    # the large scales that overflow under a finite band
    for w_v, wn_v in ((BIG, -BIG), (BIG, INF), (-BIG, 0.5 * BIG), (1e31, -INF)):
        w, wn, parts = _case(20001, 70, [torch.float32])
        w[7], wn[7] = w_v, wn_v
        cases.append((w, wn, parts, tau))
    _check(lib, cases)
    _check(lib, cases, skip=1)
