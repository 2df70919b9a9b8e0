"""Kernels whose lanes share LDS, run on the CPU lane by lane with no order but their own meeting
points (``csrc/host_check/lanes``): what a lane reads of another lane's must have been ordered by
the kernel, not by the way the compiler happened to place it. Bit for bit against the oracle."""

from __future__ import annotations

import hashlib
import shutil
import subprocess
from pathlib import Path

import pytest

import oracle as O

CHECK = Path(__file__).resolve().parent.parent / "pots-2.0_amd" / "csrc" / "host_check"


@pytest.fixture(scope="module")
def tree_lanes() -> Path:
    if shutil.which("make") is None or not Path("/opt/rocm/llvm/bin/clang++").exists():
        pytest.skip("needs make and clang++")
    r = subprocess.run(["make", "-C", str(CHECK), "_build/tree_lanes"], capture_output=True,
                       text=True, timeout=300)
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-2000:]
    return CHECK / "_build" / "tree_lanes"


@pytest.mark.parametrize("order", ([], ["last-first"]))
@pytest.mark.parametrize("n", [1, 2, 3, 129, 255, 256, 257, 513])  # one turn a quad, two; two tiles
def test_outer_tree_orders_its_lanes(tree_lanes, n, order):
    leaves = [hashlib.sha256(i.to_bytes(4, "little")).digest() for i in range(n)]
    r = subprocess.run([str(tree_lanes), str(n), *order], input=b"".join(leaves),
                       capture_output=True, timeout=120)
    assert r.returncode == 0, r.stderr
    assert r.stdout == O.merkle_tree(leaves)
