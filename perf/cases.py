"""The contractions that performance is measured on.

Every case is one pass through a public entry point as a user's program calls
it: a Contraction called on its tensors (kind "gett"), the differentiable
contract() with its backward pass (kind "grad"), or one launch of a bound
GettBatch (kind "batch").  The plan, the workspace and the bound batch are
what such a program lays out once and keeps.  Index patterns are those of
tccg_amd.workloads; the listed sizes are its configurations, one ragged
variant, and drawn cases vary every extent over the ranges below.
"""
from __future__ import annotations

import math

import torch

from tccg_amd import Contraction
from tccg_amd.autograd import adjoints, contract
from tccg_amd.batch import GettBatch, group_candidates, random_batch

# name -> (C, A, B index lists, extent ranges by label); the leftmost index is
# stride-one, a torch tensor holds the reversed shape
PATTERNS = {
    "abij-ima-mjb": ("abij", "ima", "mjb", {"abij": (8, 32), "m": (8, 32)}),
    "abcd-akc-kdb": ("abcd", "akc", "kdb", {"abcd": (16, 56), "k": (16, 96)}),
    "abcd-aebf-dfce": ("abcd", "aebf", "dfce", {"abcd": (20, 72), "ef": (12, 48)}),
    "abc-akb-kc": ("abc", "akb", "kc", {"abc": (96, 384), "k": (4, 16)}),
    "abcdef-dgfa-gceb": ("abcdef", "dgfa", "gceb", {"abcdef": (10, 24), "g": (32, 96)}),
    "abcd-aklb-lckd": ("abcd", "aklb", "lckd", {"abcd": (24, 72), "kl": (8, 32)}),
}

# Relative 2-norm difference that another correct implementation at the same
# precision shows, about four times the largest measured error against 64 bits:
# f32 1.5e-6 (k = 5184), split-BF16 7.4e-7 (k = 2304, and more on the adjoints'
# k range), f64 1.9e-15, bf16 2.1e-3; FP8 e4m3 with per-tensor scales 3.7e-2,
# stated at 3e-2.
REL = {"f32": 6e-6, "bf16x3": 6e-6, "f64": 8e-15, "bf16": 8e-3, "fp8": 3e-2}


def _gett(name, pattern, prec, sizes, alpha=1.0, beta=0.0):
    case = {"kind": "gett", "pattern": pattern, "prec": prec, "alpha": alpha, "beta": beta}
    case.update(sizes)
    if name:
        case["name"] = name
    return case


def listed():
    uni = lambda labels, n: {l: n for l in labels}
    return [
        # the reference's example.tccg: the smallest calls, where launches and
        # host latency are what a caller waits for
        _gett("example 24 f32", "abij-ima-mjb", "f32", uni("abijm", 24)),
        # the reference's CPU-sized configuration: a small contraction in the
        # middle of an iterative solver
        _gett("cpu48 f32", "abcd-akc-kdb", "f32", {**uni("abcd", 48), "k": 64}),
        # the compute-bound benchmark contraction in each precision that a
        # caller chooses: plain FP32 (the default), FP64, split-BF16, BF16
        _gett("abcd-aebf-dfce f32", "abcd-aebf-dfce", "f32", {**uni("abcd", 72), **uni("ef", 48)}),
        _gett("abcd-aebf-dfce f64", "abcd-aebf-dfce", "f64", {**uni("abcd", 72), **uni("ef", 48)}),
        _gett("abcd-aebf-dfce bf16x3", "abcd-aebf-dfce", "bf16x3", {**uni("abcd", 72), **uni("ef", 48)}),
        _gett("abcd-aebf-dfce bf16", "abcd-aebf-dfce", "bf16", {**uni("abcd", 72), **uni("ef", 48)}),
        # the same pattern with odd extents and an update of C (alpha and beta
        # other than 1 and 0): no extent is a multiple of a vector or a tile
        _gett("abcd-aebf-dfce ragged f32", "abcd-aebf-dfce", "f32",
              {"a": 61, "b": 37, "c": 53, "d": 47, "e": 29, "f": 31}, 1.5, 0.5),
        # short k, the time is C's write-back
        _gett("abc-akb-kc f32", "abc-akb-kc", "f32", {**uni("abc", 384), "k": 8}),
        # the 6-D contraction of the precision study: many tiles of few
        # k-steps, short contiguous runs of C; plain FP32 and FP8
        _gett("abcdef-dgfa-gceb f32", "abcdef-dgfa-gceb", "f32", {**uni("abcdef", 24), "g": 96}),
        _gett("abcdef-dgfa-gceb fp8", "abcdef-dgfa-gceb", "fp8", {**uni("abcdef", 24), "g": 96}),
        # training: forward and both adjoints through autograd
        {"name": "grad abcd-aklb-lckd f32", "kind": "grad", "pattern": "abcd-aklb-lckd", "prec": "f32",
         **uni("abcd", 72), **uni("kl", 32)},
        # uneven contractions launched together (block-sparse tensors)
        {"name": "batch 40 f32", "kind": "batch", "n": 40, "sizes": 0, "lo": 8, "hi": 96, "step": 8},
    ]


def _cost(case):
    """Flops of one pass with the precisions weighted by their matrix rates."""
    w = work(case)
    return w["flops"] * {"f64": 2.0, "bf16x3": 0.5, "bf16": 0.1, "fp8": 0.1}.get(case.get("prec"), 1.0)


def draw(rng):
    """One more case: a pattern, its precision and every extent drawn over the
    pattern's range (log-uniform where that spans more than a factor of ten,
    as the batch size does), odd values as likely as even ones."""
    limit = max(_cost(c) for c in listed())
    while True:
        kind = rng.choice(["gett"] * 9 + ["grad"] * 2 + ["batch"])
        if kind == "batch":
            case = {"kind": "batch", "n": int(round(math.exp(rng.uniform(math.log(4), math.log(40))))),
                    "sizes": rng.randrange(1, 1 << 16), "lo": rng.choice([7, 8]), "hi": 96, "step": rng.choice([1, 8])}
        else:
            pattern = "abcd-aklb-lckd" if kind == "grad" else rng.choice(sorted(PATTERNS))
            sizes = {l: rng.randint(lo, hi) for labels, (lo, hi) in PATTERNS[pattern][3].items() for l in labels}
            precs = ["f32"] * 4 + ["f64", "bf16x3", "bf16"]
            if pattern == "abcdef-dgfa-gceb":
                precs += ["fp8"] * 2
            prec = rng.choice(precs[:6] if kind == "grad" else precs)
            if kind == "grad":
                case = {"kind": "grad", "pattern": pattern, "prec": prec, **sizes}
            else:
                alpha, beta = rng.choice([(1.0, 0.0)] * 3 + [(1.5, 0.5)])
                case = _gett(None, pattern, prec, sizes, alpha, beta)
        if _cost(case) <= limit:
            return case


def _contraction(case):
    c, a, b, _ = PATTERNS[case["pattern"]]
    return Contraction.from_labels(list(c), list(a), list(b), {l: case[l] for l in set(c + a + b)},
                                   case.get("alpha", 1.0), case.get("beta", 0.0))


def _batch(case):
    return random_batch(case["n"], case["sizes"], lo=case["lo"], hi=case["hi"], step=case["step"])


def _inputs(case, seed):
    """Operands (and what an update or a backward pass reads besides) of one
    pass: uniform[-1, 1], or N(0, 1) for the precision study and training."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    normal = case["kind"] == "grad" or case.get("pattern") == "abcdef-dgfa-gceb"
    dt = torch.float64 if case.get("prec") == "f64" else torch.float32

    def make(shape):
        if normal:
            return torch.randn(shape, dtype=dt, device="cuda", generator=g)
        return torch.rand(shape, dtype=dt, device="cuda", generator=g).mul_(2).sub_(1)

    if case["kind"] == "batch":
        ab = [(make(c.shapes()[0]), make(c.shapes()[1])) for c in _batch(case)]
        return [x for x, _ in ab], [y for _, y in ab], None
    sa, sb, sc = _contraction(case).shapes()
    A, B = make(sa), make(sb)
    # an update reads C, a backward pass the gradient of C
    third = make(sc) if case["kind"] == "grad" or case["beta"] != 0 else None
    return A, B, third


def prepare(case, seed):
    A, B, third = _inputs(case, seed)
    if case["kind"] == "batch":
        cs = _batch(case)
        tile, order, _ = group_candidates(cs)[0]
        Cs = [torch.zeros(c.shapes()[2], device="cuda") for c in cs]
        return {"kind": "batch", "C": Cs,
                "batch": GettBatch(cs, group_tile=tile, group_order=order).bind(A, B, Cs)}
    c = _contraction(case)
    c.device_plan(case["prec"])
    if case["kind"] == "grad":
        for adj in adjoints(c):
            adj.device_plan(case["prec"])
        return {"kind": "grad", "c": c, "prec": case["prec"], "A": A.requires_grad_(), "B": B.requires_grad_(),
                "dC": third}
    C = third if third is not None else torch.zeros(c.shapes()[2], dtype=A.dtype, device="cuda")
    return {"kind": "gett", "c": c, "prec": case["prec"], "A": A, "B": B, "C": C}


def run(state):
    if state["kind"] == "batch":
        state["batch"].launch()
        return state["C"]
    if state["kind"] == "grad":
        A, B = state["A"], state["B"]
        A.grad = None
        B.grad = None
        C = contract(A, B, state["c"], state["prec"])
        C.backward(state["dC"])
        return {"C": C.detach(), "dA": A.grad, "dB": B.grad}
    return state["c"](state["A"], state["B"], state["C"], prec=state["prec"])


def _sizes(c):
    n = lambda T: math.prod(i.size for i in T.indices)
    k = math.prod(i.size for i in c.A0.indices if i.label not in {j.label for j in c.C0.indices})
    return n(c.A0), n(c.B0), n(c.C0), 2.0 * n(c.C0) * k


def work(case):
    """Operands read once, results written once (C read too where beta is not
    0, the three tensors read and written for a pass with gradients)."""
    if case["kind"] == "batch":
        rows = [_sizes(c) for c in _batch(case)]
        return {"bytes": sum(4.0 * (a + b + c) for a, b, c, _ in rows), "flops": sum(f for _, _, _, f in rows)}
    a, b, c, f = _sizes(_contraction(case))
    esz = 8.0 if case["prec"] == "f64" else 4.0
    if case["kind"] == "grad":
        return {"bytes": esz * 2 * (a + b + c), "flops": 3 * f}
    return {"bytes": esz * (a + b + c * (2 if case["beta"] != 0 else 1)), "flops": f}


def tolerance(case):
    return {"rel": REL[case.get("prec", "f32")]}


def _contract64(c_l, a_l, b_l, A, B):
    """sum over the shared labels in float64; labels and tensors in TCCG order
    (a torch tensor's shape is the labels reversed), as one plain product."""
    ra, rb, rc = [x[::-1] for x in (a_l, b_l, c_l)]
    k = [l for l in ra if l in rb]
    m, n = [l for l in ra if l not in rb], [l for l in rb if l not in ra]
    P = A.double().permute([ra.index(l) for l in m + k]).contiguous()
    Q = B.double().permute([rb.index(l) for l in k + n]).contiguous()
    shape = list(P.shape[:len(m)]) + list(Q.shape[len(k):])
    kk = math.prod(P.shape[len(m):])
    R = P.reshape(-1, kk) @ Q.reshape(kk, -1)
    return R.reshape(shape).permute([(m + n).index(l) for l in rc]).contiguous()


def exact(case, seed):
    A, B, third = _inputs(case, seed)
    labels = lambda T: [i.label for i in T.indices]
    if case["kind"] == "batch":
        return [_contract64(labels(c.C0), labels(c.A0), labels(c.B0), a, b) for c, a, b in zip(_batch(case), A, B)]
    c_l, a_l, b_l = [list(x) for x in PATTERNS[case["pattern"]][:3]]
    C = _contract64(c_l, a_l, b_l, A, B)
    if case["kind"] == "grad":
        return {"C": C, "dA": _contract64(a_l, c_l, b_l, third, B), "dB": _contract64(b_l, a_l, c_l, A, third)}
    C *= case["alpha"]
    if case["beta"] != 0:
        C += case["beta"] * third.double()
    return C
