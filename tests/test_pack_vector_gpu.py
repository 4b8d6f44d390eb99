"""The pack kernel's four-element reads: both read orders (the operand's
stride-one index free or contracted), extents at which runs of four break
(odd, under four, whole), operands off the 16-byte boundary, every precision.
The packed and the unpacked kernel of one tile shape convert the same values
and add them in the same order, so their results are the same bits."""
import numpy as np
import pytest

from tccg_amd import Contraction
from tccg_amd.plan import BF16, BF16X3, F32, F64, FP8, PACKED_TILES, TILES, build_packed_plan, build_plan

from .gpu_helpers import inputs

pytestmark = pytest.mark.gpu


def _same_shape_tiles(prec):
    for tp, shape in enumerate(PACKED_TILES[prec]):
        for tu, other in enumerate(TILES[prec]):
            if tuple(shape[:3]) == tuple(other[:3]):
                return tp, tu
    pytest.skip("no tile shape in both kernels")


@pytest.mark.parametrize("prec", [F32, F64, BF16X3, BF16, FP8])
@pytest.mark.parametrize("a_l, b_l", [("akb", "ck"), ("kab", "kc"), ("bak", "kc")])
@pytest.mark.parametrize("a, b, c, k", [(4, 33, 65, 32), (3, 50, 7, 35), (64, 2, 64, 96), (129, 1, 2, 5)])
def test_pack_reads(prec, a_l, b_l, a, b, c, k):
    import torch
    con = Contraction.from_labels(list("abc"), list(a_l), list(b_l), dict(a=a, b=b, c=c, k=k))
    dtype = np.float64 if prec == F64 else np.float32
    A, B, C = inputs(con, 3, "normal", dtype)
    tp, tu = _same_shape_tiles(prec)
    plans = (build_packed_plan(con.problem, prec, tp), build_plan(con.problem, prec, tu, m_blocked=False))
    ref = None
    for off in (0, 1, 3):                     # elements off the allocation's boundary
        views = []
        for X in (A, B):
            buf = torch.full((X.size + off + 4,), float("nan"), dtype=torch.from_numpy(X).dtype, device="cuda")
            v = buf[off:off + X.size].view(X.shape)
            v.copy_(torch.from_numpy(np.ascontiguousarray(X)))
            views.append(v)
        for plan in plans[:1] if off else plans:   # the unpacked kernel's vector loads want 16-byte alignment
            out = torch.empty(C.shape, dtype=views[0].dtype, device="cuda")
            print("pack reads", prec, a_l, b_l, off, plan.describe(), flush=True)
            con.device_plan(prec, plan=plan).run(views[0], views[1], out, 1.0, 0.0)
            torch.cuda.synchronize()
            out = out.cpu().numpy()
            ref = out if ref is None else ref
            assert np.array_equal(out, ref)
