"""The framework's work as its users call it, as cases to time and to compare.

A user of this framework verifies training-step transcripts (checks 2, 5 and 6a) or commits
them on the prover's side. The kinds below are the calls such programs make, on data in HBM:

leaf     ``merkle.hash_tensor_leaf``: one tensor's leaf hash, bytes back on the host. What a
         caller of the drop-in hashing API does per tensor.
commit   ``leaves.commit_leaves_device``: the prover's commitment of a whole step, layout
         checks, hashing, Merkle tree and the tree's copy to the host.
digests  ``StepHasher.digests`` and ``merkle_tree_device``: check 2 on a resident transcript
         whose layout repeats (the plan is kept), leaf digests and tree left in HBM.
gemm     ``FvPlan.rows`` and ``verdicts`` over products of one shape: check 5 for a
         multilayer perceptron or one captured matmul, challenges keyed on a root in host
         memory. fp32 products each hold one forged entry, which is what the check is for and
         makes the residuals more than rounding noise.
layer    the same calls over every product of a decoder step, whose backward products share
         operands with others transposed (forward and backward products alike).
update   ``UpdatePlan.run``: check 6a over a block's linear weights.
step     ``DeviceStepVerifier.run``: checks 2 and 5 of one step and its verdict on the host.

Values are what the paths meet: normal weights and activations, products rounded to the
compute dtype as a step stores them, weights after an SGD step with the committed gradients.
"""

from __future__ import annotations

import math
import sys
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path.cwd() / "pots-2.0_amd"))

from setup.records import Record  # noqa: E402
from verification.commitment import native  # noqa: E402
from verification.commitment.encoding import TAG_PRODUCT, TAG_WEIGHT  # noqa: E402
from verification.commitment.leaves import StepHasher, commit_leaves_device  # noqa: E402
from verification.commitment.merkle import hash_tensor_leaf  # noqa: E402
from verification.computation.instances.decoder import DecoderComputation  # noqa: E402
from verification.prover.synthetic import synthetic_step  # noqa: E402
from verification.verifier.bands import Bands  # noqa: E402
from verification.verifier.step import DeviceStepVerifier  # noqa: E402

DEV = "cuda"
DTYPES = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16}
ETA, EPS_W = 1e-4, 2.0**-24


def _decoder_case(name, kind, dtype, **kw):
    case = {"kind": kind, "dtype": dtype, "bias": dtype == "bf16", "k": 1, **kw}
    return {"name": name, **case} if name else case


def listed():
    return [
        # one norm's gain: the smallest leaf a transcript holds, a call that is all latency
        {"name": "leaf_norm", "kind": "leaf", "dtype": "fp32", "rows": 1, "cols": 1536, "skip": 0},
        # one square weight matrix, 64 MiB: an ordinary single-tensor call
        {"name": "leaf_weight", "kind": "leaf", "dtype": "fp32", "rows": 4096, "cols": 4096,
         "skip": 0},
        # the commitment of a toy decoder's step (the size the tests use): host work, launches
        _decoder_case("commit_tiny", "commit", "bf16", L=2, d=64, d_f=128, n_h=4, n_kv=2,
                      n_v=160, n_s=2, n=32),
        # the commitment of a 135M-parameter decoder's fp32 step, 7.7 thousand leaves, 3 GB
        _decoder_case("commit_135m", "commit", "fp32", L=30, d=576, d_f=1536, n_h=9, n_kv=3,
                      n_v=49152, n_s=4, n=256),
        # check 2 on two layers of a 1.5B-parameter decoder and its head, 9 GB of leaves
        _decoder_case("digests_2layer", "digests", "bf16", L=2, d=1536, d_f=8960, n_h=12,
                      n_kv=2, n_v=151936, n_s=4, n=2048),
        # check 5 of a small perceptron's step: six fp32 products with biases, odd sizes
        {"name": "gemm_mlp", "kind": "gemm", "dtype": "fp32", "count": 6, "n": 100, "q": 390,
         "w": 257, "k": 2, "bias": True},
        # one large fp32 matmul under eight challenges (8192 x 4096 x 4096)
        {"name": "gemm_large", "kind": "gemm", "dtype": "fp32", "count": 1, "n": 8192,
         "q": 4096, "w": 4096, "k": 8, "bias": False},
        # ragged bf16 products under the sixteen challenges of the adversarial setting
        {"name": "gemm_k16", "kind": "gemm", "dtype": "bf16", "count": 8, "n": 1000, "q": 2050,
         "w": 1537, "k": 16, "bias": False},
        # check 5 of one decoder layer, forward and backward, at the 1.5B model's sizes
        _decoder_case("layer_fwd_bwd", "layer", "bf16", L=1, d=1536, d_f=8960, n_h=12, n_kv=2,
                      n_v=4096, n_s=4, n=2048) | {"k": 4},
        # check 6a over four layers' linear weights with bf16 gradients, 1.9 GB
        {"name": "update_4layer", "kind": "update", "dtype": "bf16", "L": 4, "d": 1536,
         "d_f": 8960, "kv": 256, "parts": 1},
        # checks 2 and 5 of a small decoder's step, and the verdict on the host: latency
        _decoder_case("step_tiny", "step", "bf16", L=2, d=128, d_f=512, n_h=2, n_kv=1, n_v=512,
                      n_s=2, n=128) | {"k": 4},
        # checks 2 and 5 of two layers of the 1.5B model with its head: the headline work
        _decoder_case("step_2layer", "step", "bf16", L=2, d=1536, d_f=8960, n_h=12, n_kv=2,
                      n_v=151936, n_s=4, n=2048) | {"k": 4},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_decoder(rng, kind, most):
    while True:
        d_h = rng.choice([16, 32, 64, 128])
        n_h = _log(rng, 1, 16)
        n_kv = rng.choice([g for g in range(1, n_h + 1) if n_h % g == 0])
        case = _decoder_case(None, kind, rng.choice(["fp32", "bf16", "bf16"]),
                             L=_log(rng, 1, 8), d=n_h * d_h, d_f=_log(rng, 64, 8960), n_h=n_h,
                             n_kv=n_kv, n_v=_log(rng, 100, 60000), n_s=rng.randint(1, 8),
                             n=_log(rng, 16, 2048))
        case["k"] = rng.choice([1, 2, 4, 4, 5, 16])
        if work(case)["bytes"] <= most:
            return case


def draw(rng):
    kind = rng.choice(["leaf", "commit", "digests", "gemm", "gemm", "layer", "update", "step",
                       "step"])
    if kind == "leaf":
        rows = _log(rng, 1, 16384)
        return {"kind": kind, "dtype": rng.choice(["fp32", "bf16", "fp16"]), "rows": rows,
                "cols": _log(rng, 1, 16384), "skip": rng.choice([0, 0, 0, 1])}
    if kind == "gemm":
        dtype = rng.choice(["fp32", "bf16"])
        while True:
            case = {"kind": kind, "dtype": dtype, "count": _log(rng, 1, 64),
                    "n": _log(rng, 1, 16384), "q": _log(rng, 8, 16384), "w": _log(rng, 1, 16384),
                    "k": rng.choice([1, 2, 4, 5, 8, 16]), "bias": rng.random() < 0.3}
            if work(case)["bytes"] <= 1.5e9:
                return case
    if kind == "update":
        while True:
            case = {"kind": kind, "dtype": rng.choice(["fp32", "bf16"]), "L": _log(rng, 1, 8),
                    "d": _log(rng, 32, 4096), "d_f": _log(rng, 64, 8960),
                    "kv": _log(rng, 16, 1024), "parts": rng.choice([1, 1, 2, 4])}
            if work(case)["bytes"] <= 3e9:
                return case
    return _draw_decoder(rng, kind, 1.5e9)


# ---- the work a path cannot do without ------------------------------------------------------

def _esz(dtype):
    return 4 if dtype == "fp32" else 2


def _computation(case):
    return DecoderComputation(L=case["L"], d=case["d"], d_f=case["d_f"], n_h=case["n_h"],
                              n_kv=case["n_kv"], n_v=case["n_v"], n_s=case["n_s"], n=case["n"],
                              qkv_bias=case["bias"], compute_dtype=DTYPES[case["dtype"]])


def _leaf_bytes(case):
    """Message bytes, digests and tree nodes of a decoder step's leaves."""
    L, d, d_f, n = case["L"], case["d"], case["d_f"], case["n"]
    c = _computation({**case, "n_s": 1, "L": 1})
    q, kv, N, e = d, c.n_kv * c.d_h, case["n_s"] * n, _esz(case["dtype"])
    layer_w = (q + 2 * kv) * d + d * q + 3 * d * d_f
    weights = case["n_v"] * d + L * layer_w
    out = q + 2 * kv + d + 2 * d_f + d             # columns of a layer's forward products
    back = 3 * d + q + 2 * d + d_f                 # and of its input gradients
    members = case["n_s"] * case["n_h"]
    prods = L * (N * (out + back) + layer_w + members * (2 * n * n + 4 * n * c.d_h)) + \
        N * case["n_v"] + N * d + case["n_v"] * d
    count = case["n_s"] + 2 * (12 * L + 2) + L * (21 + 6 * members) + 3
    return 12 * N + 8 * weights + e * prods + 96 * count


def _operand_work(case):
    """Bytes of A (one read where two products share it transposed), B and P, and flops."""
    L, d, d_f, n, n_v = case["L"], case["d"], case["d_f"], case["n"], case["n_v"]
    c = _computation({**case, "n_s": 1, "L": 1})
    N, dh, kv = case["n_s"] * n, c.d_h, c.n_kv * c.d_h
    linears = [(d, d), (kv, d), (kv, d), (d, d), (d_f, d), (d_f, d), (d, d_f)]  # (out, in)
    a = b = p = vec = 0
    for mult, o, i in [(L, o, i) for o, i in linears] + [(1, n_v, d)]:
        a += mult * (N * i + N * o)          # inputs; output gradients, shared with G's A
        b += mult * (2 * o * i + N * i)
        p += mult * (N * o + N * i + o * i)
        vec += mult * (3 * N * i + 3 * N * o + 3 * o * i)
    members = L * case["n_s"] * case["n_h"]
    a += members * (2 * n * dh + 2 * n * n)
    b += members * 6 * n * dh
    p += members * (2 * n * n + 4 * n * dh)
    vec += members * (6 * n * n + 12 * n * dh)
    return _esz(case["dtype"]) * a, _esz(case["dtype"]) * b, _esz(case["dtype"]) * p, \
        2.0 * case["k"] * vec


def work(case):
    kind = case["kind"]
    if kind == "leaf":
        return {"bytes": case["rows"] * case["cols"] * _esz(case["dtype"]) + 32, "flops": 0}
    if kind in ("commit", "digests"):
        return {"bytes": _leaf_bytes(case), "flops": 0}
    if kind == "gemm":
        n, q, w = case["n"], case["q"], case["w"]
        area = case["count"] * (n * q + q * w + n * w)
        return {"bytes": _esz(case["dtype"]) * area, "flops": 2.0 * case["k"] * area}
    if kind == "update":
        n = _update_entries(case)
        return {"bytes": n * (8 + case["parts"] * _esz(case["dtype"])),
                "flops": n * (7 + case["parts"])}
    a, b, p, flops = _operand_work(case)
    if kind == "layer":
        return {"bytes": a + b + p, "flops": flops}
    return {"bytes": _leaf_bytes(case) + a + b, "flops": flops}  # step: P is read as a leaf


def _update_shapes(case):
    d, d_f, kv = case["d"], case["d_f"], case["kv"]
    return [(d, d), (kv, d), (kv, d), (d, d), (d_f, d), (d_f, d), (d, d_f)] * case["L"]


def _update_entries(case):
    return sum(o * i for o, i in _update_shapes(case))


# ---- what a program has in hand before the call ---------------------------------------------

def _root(seed):
    return bytes((seed * 7 + 13 * i + 1) & 0xFF for i in range(32))


def _random_leaves(c, seed):
    """A step's leaves in layout order, its products' values drawn instead of multiplied."""
    g = torch.Generator(device=DEV).manual_seed(seed)
    host = torch.Generator().manual_seed(seed)
    leaves = []
    for _ in range(c.n_s):
        ids = torch.randint(0, c.n_v, (c.n,), generator=host, dtype=torch.int32)
        leaves.append(Record(ids, torch.roll(ids, -1), torch.ones(c.n, dtype=torch.int32)))

    def weights():
        return [torch.randn(c.weight_shapes[x], generator=g, device=DEV).mul_(0.02)
                for x in c.weight_names]

    leaves += weights()
    leaves += [torch.randn(s.p_shape, generator=g, device=DEV, dtype=c.product_dtype)
               for s in c.products]
    return leaves + weights()


def _gemm_operands(case, seed):
    """``(a, b, p, bias)`` of each product; P rounded to the compute dtype from fp32 sums."""
    g = torch.Generator(device=DEV).manual_seed(seed)
    dt, n, q, w = DTYPES[case["dtype"]], case["n"], case["q"], case["w"]
    out = []
    for _ in range(case["count"]):
        a = torch.randn(n, q, generator=g, device=DEV).to(dt)
        b = torch.randn(q, w, generator=g, device=DEV).mul_(q ** -0.5).to(dt)
        p = a.float() @ b.float()
        bias = None
        if case["bias"]:
            bias = torch.randn(w, generator=g, device=DEV).to(dt).float()
            p += bias
        if case["dtype"] == "fp32":
            at = int(torch.randint(0, n * w, (1,), generator=g, device=DEV))
            p.view(-1)[at] += 64.0
        out.append((a, b, p.to(dt), bias))
    return out


def _layer_operands(case, seed):
    c = _computation(case)
    step = synthetic_step(c, seed=seed, device=DEV)
    out = []
    for spec in c.products:
        a, b = step.operands[spec.m]
        bias = step.w_t(spec.bias).to(c.operand_dtype).float() if spec.bias else None
        out.append((a, b, step.product(spec.m), bias))
    return c, step, out


def _check5(state, ops, case):
    """The plan and the verdict table of check 5 over ``ops``."""
    lib = native.get()
    prods = [native.FvProduct(a, b, p, m, bias) for m, (a, b, p, bias) in enumerate(ops, 1)]
    state["plan"] = lib.fv_plan(prods, case["k"])
    bands = Bands.provisional()
    state["specs"] = native.verdict_specs(
        [a.shape[1] + (bias is not None) for a, _, _, bias in ops],
        [a.shape[0] for a, _, _, _ in ops], [bias is not None for _, _, _, bias in ops],
        [bands.kappa_max] * len(ops))
    state["tau"] = bands.tau
    state["ops"] = ops
    return state


def prepare(case, seed):
    kind = case["kind"]
    state = {"kind": kind, "case": case, "root": _root(seed)}
    if kind == "leaf":
        g = torch.Generator(device=DEV).manual_seed(seed)
        rows, cols, skip = case["rows"], case["cols"], case["skip"]
        flat = torch.randn(rows * cols + skip, generator=g, device=DEV).to(DTYPES[case["dtype"]])
        shape = (cols,) if rows == 1 else (rows, cols)
        return state | {"t": flat[skip:].view(shape),
                        "tag": TAG_WEIGHT if case["dtype"] == "fp32" else TAG_PRODUCT}
    if kind in ("commit", "digests"):
        c = _computation(case)
        leaves = _random_leaves(c, seed)
        if kind == "commit":
            return state | {"c": c, "leaves": leaves}
        return state | {"hasher": StepHasher(c, leaves), "leaves": leaves}
    if kind == "gemm":
        return _check5(state, _gemm_operands(case, seed), case)
    if kind == "layer":
        _, step, ops = _layer_operands(case, seed)
        return _check5(state | {"step": step}, ops, case)
    if kind == "update":
        g = torch.Generator(device=DEV).manual_seed(seed)
        dt, weights = DTYPES[case["dtype"]], []
        for shape in _update_shapes(case):
            w = torch.randn(shape, generator=g, device=DEV).mul_(0.02)
            parts = [torch.randn(shape, generator=g, device=DEV).to(dt)
                     for _ in range(case["parts"])]
            grad = parts[0].float()
            for x in parts[1:]:
                grad = grad + x.float()
            weights.append(native.UpdateWeight(w, torch.add(w, grad, alpha=-ETA), parts,
                                               Bands.provisional().tau_w))
        return state | {"plan": native.get().update_plan(weights, ETA, EPS_W)}
    c, step, ops = _layer_operands(case, seed)
    v = DeviceStepVerifier(c, step.leaves, lambda spec: step.operands[spec.m], k=case["k"])
    return state | {"step": step, "verifier": v, "ops": ops,
                    "root": commit_leaves_device(c, step.leaves).root}


# ---- one pass -------------------------------------------------------------------------------

def _row_parts(case, rows):
    """A row table by column: the sums each under their own scale, the residuals together.
    The residuals of honest fp32 products are rounding noise, so their rows stay in one piece."""
    if case["dtype"] == "fp32" and case["kind"] != "gemm":
        return {"rows": rows}
    out = {name: rows[:, i] for i, name in enumerate(("nu", "p_abs", "p_norm", "u2", "b2"))}
    return out | {"residual": rows[:, 5:]}


def run(state):
    kind, case = state["kind"], state["case"]
    if kind == "leaf":
        return np.frombuffer(hash_tensor_leaf(state["tag"], state["t"]), dtype=np.uint8)
    if kind == "commit":
        return np.frombuffer(commit_leaves_device(state["c"], state["leaves"]).root,
                             dtype=np.uint8)
    if kind == "digests":
        digests, bad = state["hasher"].digests()
        return {"digests": digests, "bad": bad,
                "nodes": native.get().merkle_tree_device(digests)}
    if kind in ("gemm", "layer"):
        rows = state["plan"].rows(state["root"])
        codes, _, first = native.get().verdicts(
            rows, state["specs"], k=case["k"], eps_in=_eps(case), eps_acc=2.0**-24,
            tau=state["tau"])
        return {"codes": codes, "first": first, **_row_parts(case, rows)}
    if kind == "update":
        return state["plan"].run()
    v = state["verifier"].run(state["root"])
    return {"root": np.frombuffer(v.root, dtype=np.uint8), "bad": v.first_bad,
            "fail": v.first_fail, "codes": v.codes, **_row_parts(case, v.rows)}


def _eps(case):
    return 2.0**-24 if case["dtype"] == "fp32" else 2.0**-8


# ---- what results may differ by -------------------------------------------------------------

def tolerance(case):
    """Hashes, trees, verdict codes and check 6a's maxima are exact. Check 5's sums are fp32
    sums of non-negative terms (measured against 64 bits: up to 2e-6). Its residuals are
    differences of fp32 sums: a forged fp32 entry leaves 64 times a challenge (measured up to
    2e-5, where that challenge is small), a bf16 product its rounding (up to 1.3e-5 at the
    smallest step, more for a product of few entries)."""
    if case["kind"] in ("leaf", "commit", "digests", "update"):
        return "exact"
    rel = 1e-5 if case["dtype"] == "fp32" and case["kind"] != "gemm" else 4e-4
    return {"rel": rel, "max": 10 * rel, "differ": 0.0}


# ---- the same in 64 bits --------------------------------------------------------------------

_PERM = (2, 6, 3, 10, 7, 0, 4, 13, 1, 11, 12, 5, 9, 14, 15, 8)
_IV = (0x6A09E667, 0xBB67AE85, 0x3C6EF372, 0xA54FF53A, 0x510E527F, 0x9B05688C, 0x1F83D9AB,
       0x5BE0CD19)
_QUADS = ((0, 4, 8, 12), (1, 5, 9, 13), (2, 6, 10, 14), (3, 7, 11, 15),
          (0, 5, 10, 15), (1, 6, 11, 12), (2, 7, 8, 13), (3, 4, 9, 14))


def _challenges(root, m, k, width):
    """Product ``m``'s challenge matrix ``[width, k]`` in fp64: the keyed BLAKE3 output stream
    of ``0x10 ‖ m ‖ j``, one compression per 16 entries, on int64 lanes."""
    mask, blocks = 0xFFFFFFFF, (width + 15) // 16
    t = torch.arange(blocks, device=DEV, dtype=torch.int64).repeat_interleave(k)
    j = torch.arange(1, k + 1, device=DEV, dtype=torch.int64).repeat(blocks)
    zero = torch.zeros_like(t)
    label = 0x10 | (m >> 24 & 255) << 8 | (m >> 16 & 255) << 16 | (m >> 8 & 255) << 24
    msg = [zero + label, (m & 255) + (j << 8)] + [zero] * 14
    key = [int.from_bytes(root[4 * i:4 * i + 4], "little") for i in range(8)]
    v = [zero + x for x in (*key, *_IV[:4])] + [t, zero, zero + 6, zero + (1 | 2 | 8 | 16)]

    def rot(x, r):
        return (x >> r | x << (32 - r)) & mask

    for r in range(7):
        for i, (a, b, c, d) in enumerate(_QUADS):
            for x, s0, s1 in ((msg[2 * i], 16, 12), (msg[2 * i + 1], 8, 7)):
                v[a] = (v[a] + v[b] + x) & mask
                v[d] = rot(v[d] ^ v[a], s0)
                v[c] = (v[c] + v[d]) & mask
                v[b] = rot(v[b] ^ v[c], s1)
        msg = [msg[i] for i in _PERM]
    words = [v[i] ^ v[i + 8] for i in range(8)] + [v[i + 8] ^ key[i] for i in range(8)]
    w = torch.stack(words, 1).view(blocks, k, 16).transpose(1, 2).reshape(16 * blocks, k)
    return ((2 * (w >> 8) + 1 - (1 << 24)).double() / 2.0**24)[:width]


def _row64(a, b, p, bias, r):
    """One product's row in 64 bits, its operands widened some rows at a time."""
    def blocks(t):
        step = max(1, (1 << 26) // max(1, t.shape[1]))
        return (t[i:i + step].double() for i in range(0, t.shape[0], step))

    b1 = torch.cat([x.abs().sum(1) for x in blocks(b)])
    b2 = torch.cat([x.square().sum(1) for x in blocks(b)])
    br = torch.cat([x @ r for x in blocks(b)])
    nu = torch.cat([x.abs() @ b1 for x in blocks(a)])
    u2 = sum((x.square() @ b2).sum() for x in blocks(a))
    ab = torch.cat([x @ br for x in blocks(a)])
    bb = torch.zeros((), device=DEV, dtype=torch.float64)
    if bias is not None:
        d = bias.double()
        nu, ab, bb = nu + d.abs().sum(), ab + d @ r, d.square().sum()
    pr = torch.cat([x @ r for x in blocks(p)])
    p1 = torch.cat([x.abs().sum(1) for x in blocks(p)])
    pq = sum(x.square().sum() for x in blocks(p))
    return torch.cat([torch.stack([nu.norm(), p1.norm(), pq.sqrt(), u2, bb]),
                      (ab - pr).norm(dim=0)])


def exact(case, seed):
    if case["kind"] not in ("gemm", "layer", "step"):
        return None
    state = prepare(case, seed)
    root, ops = state["root"], state["ops"]
    rows = torch.stack([_row64(a, b, p, bias, _challenges(root, m, case["k"], p.shape[1]))
                        for m, (a, b, p, bias) in enumerate(ops, 1)])
    names = ("root", "bad", "fail", "codes") if case["kind"] == "step" else ("codes", "first")
    return dict.fromkeys(names) | _row_parts(case, rows)
