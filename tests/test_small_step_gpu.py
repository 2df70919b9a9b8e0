"""Steps on both sides of the line from which the leaf plan is fused with the Freivalds plan
(``step.FUSE_LEAST``): the default's verdict, root and codes equal the unfused plan's, an honest
step and one with a forged product, and a caller that asks for either gets it. The rows' sums are relative 1e-6, as the fused plan's tests
hold them: the two plans take P's sums in different orders."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


def _verifiers(n, forged, fuse):
    """A step's verifiers at each of ``fuse``, and its root."""
    from verification.commitment.leaves import commit_leaves_device
    from verification.computation.instances.decoder import DecoderComputation
    from verification.prover.synthetic import synthetic_step
    from verification.verifier.step import DeviceStepVerifier
    # 31,352 chunks at n = 64, 34,680 at 128
    c = DecoderComputation(L=1, d=512, d_f=1024, n_h=4, n_kv=2, n_v=1024, n_s=2, n=n,
                           qkv_bias=True, compute_dtype=torch.bfloat16)
    step = synthetic_step(c, seed=5, operands=True)
    if forged:
        step.product(c.products[7].m).view(-1)[11] += 64.0
    return [DeviceStepVerifier(c, step.leaves, lambda s: step.operands[s.m], k=4, fuse=f)
            for f in fuse], commit_leaves_device(c, step.leaves).root


def _same(a, b, root, forged):
    assert a.root == b.root == root
    assert (a.first_bad, a.first_fail, a.check) == (b.first_bad, b.first_fail, b.check)
    assert a.check == ("5" if forged else None)
    assert torch.equal(a.codes, b.codes)
    assert torch.allclose(a.rows[:, :5], b.rows[:, :5], rtol=1e-6, atol=0)


@pytest.mark.parametrize("n", [64, 128])  # either side of the line
@pytest.mark.parametrize("forged", [False, True])
def test_fuse_as_asked(lib, n, forged):
    (on, off), root = _verifiers(n, forged, (True, False))
    assert on.fused > 0 and off.fused == 0
    for _ in range(2):
        _same(on.run(root), off.run(root), root, forged)


@pytest.mark.parametrize("n, fused", [(64, False), (128, True)])
@pytest.mark.parametrize("forged", [False, True])
def test_small_steps_are_not_fused(lib, n, fused, forged):
    from verification.commitment.leaves import commit_leaves_device
    from verification.computation.instances.decoder import DecoderComputation
    from verification.prover.synthetic import synthetic_step
    from verification.verifier.step import DeviceStepVerifier
    # 31,352 and 34,680 chunks
    c = DecoderComputation(L=1, d=512, d_f=1024, n_h=4, n_kv=2, n_v=1024, n_s=2, n=n,
                           qkv_bias=True, compute_dtype=torch.bfloat16)
    step = synthetic_step(c, seed=5, operands=True)
    if forged:
        step.product(c.products[7].m).view(-1)[11] += 64.0
    root = commit_leaves_device(c, step.leaves).root
    got = DeviceStepVerifier(c, step.leaves, lambda s: step.operands[s.m], k=4)
    plain = DeviceStepVerifier(c, step.leaves, lambda s: step.operands[s.m], k=4, fuse=False)
    assert (got.fused > 0) == fused and plain.fused == 0
    for _ in range(2):
        a, b = got.run(root), plain.run(root)
        assert a.root == b.root == root
        assert (a.first_bad, a.first_fail, a.check) == (b.first_bad, b.first_fail, b.check)
        assert a.check == ("5" if forged else None)
        assert torch.equal(a.codes, b.codes)
        assert torch.allclose(a.rows[:, :5], b.rows[:, :5], rtol=1e-6, atol=0)
