"""Tensors that start at any element: A, B and C each one element past the
16-byte boundary, and all three, for every kind of plan that reads or writes
16 bytes at a time.  The tables, tiles and order of sums are those of aligned
tensors: the same bits with beta == 0, with beta != 0 the roundings of
alpha * sum, beta * C and their sum apart (three of each, in either)."""
import numpy as np
import pytest

from tccg_amd import Contraction, codegen
from tccg_amd.plan import (BF16, BF16X3, F32, F64, FP8, FREE4, KDIM4, build_packed_plan, build_plan,
                           build_vector_plan, call_plan)
from tccg_amd.runtime import GeneratedGett
from tccg_amd.workloads import WORKLOADS

from .gpu_helpers import inputs

pytestmark = pytest.mark.gpu


def _con(c_l, a_l, b_l, **ext):
    return Contraction.from_labels(list(c_l), list(a_l), list(b_l), ext)


FREE = _con("abc", "akb", "ck", a=64, b=5, c=68, k=36)           # both FREE4
ALONG_K = _con("abc", "kab", "kc", a=24, b=9, c=33, k=44)        # both KDIM4
SHORT = _con("abc", "akb", "kc", a=96, b=40, c=37, k=8)
RUNS = _con("abc", "akc", "kb", a=64, b=128, c=4, k=40)          # C's runs span m and n, over whole tiles
LONG = _con("abc", "akc", "kb", a=64, b=256, c=16, k=4096)       # the same, k cut into pieces
# contractions whose default call was a packed plan before it became a gather one
EXAMPLE = _con("abcd", "ebad", "ce", a=24, b=24, c=24, d=24, e=24)
NEIGHBOUR = _con("abcd", "ebad", "ce", a=20, b=20, c=20, d=20, e=20)

PLANS = {
    "call": lambda c, p: call_plan(c.problem, p),
    "gather": lambda c, p: build_plan(c.problem, p, 1 if p != F32 else 0, m_blocked=False),
    "persistent": lambda c, p: build_plan(c.problem, p, 1 if p != F32 else 0, persistent=True),
    "stream": lambda c, p: build_plan(c.problem, p, 10, stream=True),
    "vector": lambda c, p: build_vector_plan(c.problem, p, 0),
    "store waves": lambda c, p: build_packed_plan(c.problem, p, {F32: 4, BF16X3: 4}.get(p, 0), store_waves=True),
    "one tile": lambda c, p: build_packed_plan(c.problem, p, 0),
    "stream-k": lambda c, p: build_packed_plan(c.problem, p, 0, stream_k=1),
}


def _moved(x, off):
    """x on the GPU, `off` elements past an allocation's start, NaN around it."""
    import torch
    buf = torch.full((x.size + off + 4,), float("nan"), dtype=torch.from_numpy(x).dtype, device="cuda")
    v = buf[off:off + x.size].view(x.shape)
    v.copy_(torch.from_numpy(np.ascontiguousarray(x)))
    return v, buf


def _check(con, run, dtype):
    import torch
    A, B, C = inputs(con, 5, "normal", dtype, with_c=True)
    eps = np.finfo(dtype).eps
    ref = {}
    for offs in ((0, 0, 0), (1, 0, 0), (0, 1, 0), (0, 0, 1), (1, 1, 1)):
        for alpha, beta in ((1.5, 0.0), (1.5, -0.75)):
            (a, _), (b, _), (c, buf) = (_moved(x, o) for x, o in zip((A, B, C), offs))
            run(a, b, c, alpha, beta)
            torch.cuda.synchronize()
            out = c.cpu().numpy()
            assert bool(buf[:offs[2]].isnan().all()) and bool(buf[offs[2] + C.size:].isnan().all())   # nothing beside C
            ref.setdefault(beta, out)
            if beta == 0:
                assert np.array_equal(out, ref[beta]), offs
            else:
                assert (np.abs(out - ref[beta]) <= 6 * eps * (np.abs(ref[0.0]) + np.abs(beta * C))).all(), offs


@pytest.mark.parametrize("con, kind, precs", [
    (EXAMPLE, "call", (F32, F64, BF16X3, BF16, FP8)), (NEIGHBOUR, "call", (F32, F64, BF16X3, BF16, FP8)),
    (FREE, "call", (F32, BF16)), (SHORT, "call", (F32, F64)), (RUNS, "call", (F32, BF16X3)),
    (FREE, "gather", (F32, F64, BF16X3, BF16, FP8)), (ALONG_K, "gather", (F32, F64, BF16X3, BF16, FP8)),
    (FREE, "persistent", (F32, BF16)), (SHORT, "stream", (F32,)), (SHORT, "vector", (F32, F64)),
    (FREE, "store waves", (F32, BF16X3, BF16)), (RUNS, "store waves", (F32, BF16)),
    (FREE, "one tile", (F32, F64)), (RUNS, "one tile", (F32, F64, BF16X3)), (LONG, "stream-k", (F32, BF16)),
])
def test_tensors_off_the_16_byte_boundary(con, kind, precs):
    for prec in precs:
        plan = PLANS[kind](con, prec)
        print("unaligned", prec, kind, plan.describe(), flush=True)
        dp = con.device_plan(prec, plan=plan) if kind != "call" else con.device_plan(prec)
        if kind == "gather":
            assert plan.modeA in (FREE4, KDIM4) and plan.modeB in (FREE4, KDIM4)
        if con in (RUNS, LONG) and kind != "call":
            assert plan.cvec or plan.crun[0]
        _check(con, dp.run, np.float64 if prec == F64 else np.float32)


@pytest.mark.parametrize("wl", ["example", "cpu48"])
def test_generated_libraries_off_the_16_byte_boundary(wl):
    con = Contraction.from_tccg(WORKLOADS[wl])
    g = GeneratedGett(codegen.GENERATED_DIR / ("lib%s.so" % codegen.workload_library_name(wl, F32)))
    print("unaligned", wl, g.info, flush=True)
    _check(con, g, np.float32)
