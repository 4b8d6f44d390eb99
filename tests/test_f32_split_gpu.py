"""FP32 contractions on the BF16 MFMAs against FP64: accuracy at least the FP32
MFMA's, and FP32's results where an operand holds values that the three parts
do not (infinities, NaNs, the extremes of the range)."""
import numpy as np
import pytest

from tccg_amd import Contraction
from tccg_amd.plan import BF16X3, F32, PACKED_TILES, build_packed_plan

from .gpu_helpers import inputs, run_gpu

pytestmark = pytest.mark.gpu

WALKS = (dict(), dict(persistent=True), dict(stream_k=1))


def _matmul(m, n, k):
    return Contraction.from_labels(["m", "n"], ["k", "m"], ["n", "k"], {"m": m, "n": n, "k": k})


def _split(c, tile, **kw):
    p = build_packed_plan(c.problem, BF16X3, tile, **kw)
    p.guard = True
    return p


def _exact(A, B, C, alpha, beta):
    """alpha A B + beta C in FP64 and the sum of the magnitudes behind each element."""
    a, b = A.astype(np.float64), B.astype(np.float64)
    with np.errstate(all="ignore"):
        return (alpha * (a @ b).T + beta * C, abs(alpha) * (np.abs(a) @ np.abs(b)).T + abs(beta * C))


def _specials(A, B):
    A, B = A.copy(), B.copy()
    A[5, 7], A[-2, -1], A[130, 33], A[70, 3] = np.inf, np.nan, 3.0e38, 1e-39
    A[40, :] *= 2.0 ** -120
    B[1, 20], B[-1, 100], B[4, 65], B[:, 3] = -np.inf, 1e-35, 2.0 ** 60, B[:, 3] * np.float32(2.0 ** -110)
    return A, B


@pytest.mark.parametrize("tile", range(len(PACKED_TILES[BF16X3])))
@pytest.mark.parametrize("walk", range(3))
def test_special_values_give_the_fp32_result(tile, walk):
    """Ragged tiles (m, n and k no multiple of any tile or pack block).  A
    worst-case bound for k rounded or truncated FP32 additions of products:
    (k + 8) 2^-23 times the sum of the magnitudes (+ the denormal range)."""
    m, n, k = 333, 290, 104
    c = _matmul(m, n, k)
    A, B, C = inputs(c, 11 + tile, with_c=True)          # torch shapes (m, k), (k, n), (n, m)
    plan = _split(c, tile, **WALKS[walk])
    print(plan.describe(), flush=True)
    for a, b in ((A, B), _specials(A, B), (A, B)):
        out = run_gpu(c, a, b, C, prec=F32, alpha=1.5, beta=0.5, plan=plan)
        fp32 = run_gpu(c, a, b, C, prec=F32, alpha=1.5, beta=0.5, plan=build_packed_plan(c.problem, F32, 2))
        ref, mag = _exact(a, b, C, 1.5, 0.5)
        assert np.array_equal(np.isnan(out), np.isnan(fp32))
        inf = np.isinf(fp32)
        assert np.array_equal(np.isinf(out), inf) and np.array_equal(out[inf], fp32[inf])
        ok = np.isfinite(out)
        bound = (k + 8) * 2.0 ** -23 * mag[ok] + 2.0 ** -125
        assert np.all(np.abs(out[ok] - ref[ok]) <= bound)


@pytest.mark.parametrize("k", [32, 100, 2304])
@pytest.mark.parametrize("dist", ["uniform", "normal"])
def test_error_no_larger_than_the_fp32_kernels(k, dist):
    c = _matmul(384, 320, k)
    A, B, C = inputs(c, k, dist)
    ref, _ = _exact(A, B, C, 1.0, 0.0)
    err = lambda plan: np.linalg.norm(run_gpu(c, A, B, C, prec=F32, plan=plan) - ref) / np.linalg.norm(ref)
    split, fp32 = err(_split(c, 0)), err(build_packed_plan(c.problem, F32, 2))
    print("k %d %s: split %.3e, FP32 MFMA %.3e" % (k, dist, split, fp32), flush=True)
    assert split <= fp32


def test_prepacked_call_and_reuse_of_a_workspace():
    """run_prepacked() after a call with raw blocks gives that call's bits, and a
    plan whose workspace has seen raw blocks gives the same bits afterwards as
    a fresh one."""
    import torch
    from tccg_amd.runtime import DevicePlan
    c = _matmul(333, 290, 104)
    A, B, _ = inputs(c, 5)
    As, Bs = _specials(A, B)
    dev = lambda x: torch.from_numpy(np.ascontiguousarray(x)).cuda()
    dp, fresh = DevicePlan(_split(c, 5)), DevicePlan(_split(c, 5))
    C = [torch.zeros(c.shapes()[2], device="cuda") for _ in range(4)]
    dp.run(dev(As), dev(Bs), C[0])
    dp.run_prepacked(C[1])
    dp.run(dev(A), dev(B), C[2])
    fresh.run(dev(A), dev(B), C[3])
    torch.cuda.synchronize()
    assert torch.equal(C[0].view(torch.int32), C[1].view(torch.int32))
    assert torch.equal(C[2], C[3])


def test_default_call_and_graph_replay():
    """The default FP32 call of a contraction that runs on the split, eager and
    replayed from a graph, between raw and plain inputs in the same buffers."""
    import torch
    c = _matmul(1500, 1400, 600)
    A, B, _ = inputs(c, 9)
    As, Bs = _specials(A, B)
    tA, tB = torch.from_numpy(A).cuda(), torch.from_numpy(B).cuda()
    tC = torch.zeros(c.shapes()[2], device="cuda")
    assert c.device_plan("f32").plan.guard
    c(tA, tB, tC)
    torch.cuda.synchronize()
    plain = tC.clone()
    g, s = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        with torch.cuda.graph(g, stream=s):
            c(tA, tB, tC)
    torch.cuda.current_stream().wait_stream(s)
    for a, b in ((As, Bs), (A, B), (As, Bs), (A, B)):
        tA.copy_(torch.from_numpy(a))
        tB.copy_(torch.from_numpy(b))
        g.replay()
        torch.cuda.synchronize()
        got = tC.clone()
        c(tA, tB, tC)
        torch.cuda.synchronize()
        assert torch.equal(got.view(torch.int32), tC.view(torch.int32))
    assert torch.equal(tC, plain)


@pytest.mark.parametrize("order", ["xcd", "lpt"])
@pytest.mark.parametrize("shape", [(128, 128, 16), (192, 192, 16), (192, 64, 16)])
def test_grouped_problems_with_special_values(shape, order):
    """A group of uneven problems, raw blocks in some operands: every problem
    against FP64 with the bound of the single call, special values as plain FP32."""
    import torch
    from tccg_amd.batch import GettBatch
    sizes = [(333, 290, 104), (64, 64, 4), (200, 131, 37), (333, 290, 104)]
    cs = [_matmul(*s) for s in sizes]
    ops = [inputs(c, 20 + i, with_c=True) for i, c in enumerate(cs)]
    ops[3] = _specials(*ops[3][:2]) + (ops[3][2],)
    alphas, betas = [1.0, 1.5, -0.5, 1.5], [0.0, 0.5, 0.0, 0.5]
    dev = lambda x: torch.from_numpy(np.ascontiguousarray(x)).cuda()
    As, Bs, Cs = ([dev(o[i]) for o in ops] for i in range(3))
    b = GettBatch(cs, alphas=alphas, betas=betas, group_tile=PACKED_TILES[F32].index(shape), group_order=order)
    assert all(p.guard for p in b.plans)
    b.bind(As, Bs, Cs).launch()
    torch.cuda.synchronize()
    for (m, n, k), (A, B, C), got, al, be in zip(sizes, ops, Cs, alphas, betas):
        out = got.cpu().numpy()
        ref, mag = _exact(A, B, C, al, be)
        fp32 = run_gpu(_matmul(m, n, k), A, B, C, prec=F32, alpha=al, beta=be,
                       plan=build_packed_plan(_matmul(m, n, k).problem, F32, 2))
        assert np.array_equal(np.isnan(out), np.isnan(fp32)) and np.array_equal(np.isinf(out), np.isinf(fp32))
        ok = np.isfinite(out)
        assert np.all(np.abs(out[ok] - ref[ok]) <= (k + 8) * 2.0 ** -23 * mag[ok] + 2.0 ** -125)


@pytest.mark.parametrize("kw", [dict(), dict(persistent=True), dict(stream_k=1)])
def test_sums_over_c_are_unbiased(kw):
    """The sum of the errors over all of C, and over each of its rows and columns,
    within five standard deviations of independent errors (their standard
    deviation times the root of their count): a rounding to one side would leave
    it, by the root of the count."""
    m, n, k = 1000, 900, 240
    c = _matmul(m, n, k)
    A, B, C = inputs(c, 3)
    plan = _split(c, 0, **kw)
    out = run_gpu(c, A, B, C, prec=F32, plan=plan).astype(np.float64)
    d = out - _exact(A, B, C, 1.0, 0.0)[0]
    sd = d.std()
    for axis in (None, 0, 1):
        s = d.sum(axis=axis)
        count = d.size if axis is None else d.shape[axis]
        assert np.all(np.abs(s) <= 5 * sd * np.sqrt(count)), (axis, np.abs(s).max() / (sd * np.sqrt(count)))
