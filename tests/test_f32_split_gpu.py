"""FP32 contractions on the BF16 MFMAs against FP64: accuracy at least the FP32
MFMA's, and FP32's results where an operand holds values that the three parts
do not (infinities, NaNs, the extremes of the range)."""
import numpy as np
import pytest

from tccg_amd import Contraction
from tccg_amd.plan import BF16X3, F32, PACKED_TILES, SPLIT_RESIDENT, build_packed_plan

from .gpu_helpers import inputs, run_gpu

pytestmark = pytest.mark.gpu

WALKS = (dict(), dict(persistent=True), dict(stream_k=1))


def _matmul(m, n, k):
    return Contraction.from_labels(["m", "n"], ["k", "m"], ["n", "k"], {"m": m, "n": n, "k": k})


def _split(c, tile, **kw):
    return build_packed_plan(c.problem, BF16X3, tile, guard=True, **kw)


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
    A[200, 40:], B[70:, 200] = 2.0 ** 40, -2.0 ** 41
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


def _words(dp):
    """(whether the last call packed a raw block, its pack blocks' words) of a
    guarded DevicePlan."""
    import ctypes
    import torch
    from tccg_amd.runtime import load_library
    off = load_library().tccg_f32_split_clear_offset(ctypes.byref(dp.cplan))
    n = (dp.plan.Mp // 64 + dp.plan.Np // 64) * (dp.plan.Kp // 32)
    head = dp.workspace[off:off + 16].view(torch.int32).cpu().numpy()
    return int(head[head[3] & 1]), dp.workspace[off + 256:off + 256 + 4 * n].view(torch.int32).cpu().numpy()


def test_values_of_every_size_are_held_and_raw_blocks_cost_one_call():
    """Operands over the whole range below the limit, subnormals included, have no
    raw block; a larger value, an infinity or a NaN makes its own pack block raw,
    and the next call's tiles look at no words for it."""
    import torch
    from tccg_amd.runtime import DevicePlan
    c = _matmul(200, 150, 130)
    rng = np.random.default_rng(7)
    wide = lambda s: np.ldexp(rng.uniform(-2, 2, s), rng.integers(-149, 34, s)).astype(np.float32)
    A, B = wide(c.shapes()[0]), wide(c.shapes()[1])
    dev = lambda x: torch.from_numpy(np.ascontiguousarray(x)).cuda()
    dp = DevicePlan(_split(c, 0))
    C = torch.zeros(c.shapes()[2], device="cuda")
    dp.run(dev(A), dev(B), C)
    torch.cuda.synchronize()
    any_, words = _words(dp)
    assert any_ == 0 and not words.any()
    for value in (np.inf, np.nan, 2.0 ** 36):
        As = A.copy()
        As[70, 40] = value
        dp.run(dev(As), dev(B), C)
        torch.cuda.synchronize()
        any_, words = _words(dp)
        nk = dp.plan.Kp // 32
        assert any_ == 1 and words.sum() == 1 and words[(70 // 64) * nk + 40 // 32] == 1   # A's m is the free set
        dp.run(dev(A), dev(B), C)
        torch.cuda.synchronize()
        any_, words = _words(dp)
        assert any_ == 0 and not words.any()


def _zero_inputs(c, seed, raw):
    """Whole numbers; C is zero where a row of A or a column of B is, and where
    the two halves of k cancel."""
    rng = np.random.default_rng(seed)
    sa, sb, _ = c.shapes()
    A, B = (rng.integers(-9, 10, s).astype(np.float32) for s in (sa, sb))
    k = sa[1]                                            # A (c, k, a), B (b, d, k)
    A[:, k // 2:, ::3], B[:, ::2, k // 2:] = A[:, :k // 2, ::3], -B[:, ::2, :k // 2]
    A[5], B[7] = 0, 0
    if raw:
        A[20, 3, 1] = 2.0 ** 60
    return A, B


@pytest.mark.parametrize("raw", [False, True])
@pytest.mark.parametrize("alpha", [1.5, -1.5])
def test_zeros_have_the_sign_of_the_fp32_kernel(alpha, raw):
    """The epilogues undo the sign of the packed rows: zeros come out as +0 (times
    alpha) all the same, from the direct and the run epilogue, the persistent and
    the stream-k walk, and in a group."""
    import torch
    from tccg_amd.batch import GettBatch
    c = Contraction.from_labels(list("abcd"), list("akc"), list("kdb"), dict(a=24, b=24, c=24, d=24, k=64))
    A, B = _zero_inputs(c, 2, raw)
    C = np.zeros(c.shapes()[2], np.float32)
    fp32 = run_gpu(c, A, B, C, prec=F32, alpha=alpha, plan=build_packed_plan(c.problem, F32, 2))
    assert np.count_nonzero(fp32 == 0) > fp32.size // 8
    runs = 0
    for tile, kw in [(0, {}), (6, {}), (8, {}), (0, WALKS[1]), (6, WALKS[1]), (4, WALKS[2]), (7, WALKS[2])]:
        plan = _split(c, tile, **kw)
        runs += plan.crun[0] > 0 and not plan.grid
        out = run_gpu(c, A, B, C, prec=F32, alpha=alpha, plan=plan)
        assert np.array_equal(out, fp32), plan.describe()   # whole numbers: exact
        assert np.array_equal(np.signbit(out), np.signbit(fp32)), plan.describe()
    assert runs
    dev = lambda x: torch.from_numpy(np.ascontiguousarray(x)).cuda()
    Cs = [torch.zeros(c.shapes()[2], device="cuda")]
    b = GettBatch([c], alphas=[alpha], betas=[0.0], group_tile=PACKED_TILES[F32].index((128, 128, 16)))
    b.bind([dev(A)], [dev(B)], Cs).launch()
    torch.cuda.synchronize()
    assert np.array_equal(np.signbit(Cs[0].cpu().numpy()), np.signbit(fp32))


@pytest.mark.parametrize("walk", range(3))
@pytest.mark.parametrize("where", ["few", "half", "A", "both"])
def test_raw_steps_over_long_k(walk, where):
    """More k-steps than a wave looks at together (64), raw blocks in a few, in
    half and in all of them: against FP64 with the bound of k rounded additions."""
    m, n, k = 200, 150, (2100 if walk != 1 else 250)
    c = _matmul(m, n, k)
    A, B, _ = inputs(c, 31)
    rng = np.random.default_rng(5)
    if where == "few":
        A[7, 5], A[150, k - 1], B[k // 2, 3] = 2.0 ** 50, -2.0 ** 45, 2.0 ** 47
    elif where == "half":
        A[:, rng.permutation(-(-k // 32))[:k // 64] * 32] *= np.float32(2.0 ** 45)
    else:
        A *= np.float32(2.0 ** 45)
        if where == "both":
            B *= np.float32(2.0 ** 45)
    for tile in SPLIT_RESIDENT:
        plan = _split(c, tile, **WALKS[walk])
        print(plan.describe(), flush=True)
        out = run_gpu(c, A, B, np.zeros(c.shapes()[2], np.float32), prec=F32, plan=plan)
        ref, mag = _exact(A, B, np.zeros(c.shapes()[2], np.float32), 1.0, 0.0)
        assert np.all(np.abs(out - ref) <= (k + 8) * 2.0 ** -23 * mag)


@pytest.mark.parametrize("ea, eb", [(-62, -62), (-63, -63), (-99, -20), (-120, 0), (-140, 14), (-65, -65)])
def test_products_at_the_bottom_of_the_range(ea, eb):
    """Held operands whose products lie around FP32's smallest normal number: the
    low products of the parts must not be lost.  The error is at most the FP32
    kernel's, but for one rounding to a subnormal result (2^-150)."""
    c = _matmul(128, 128, 64)
    rng = np.random.default_rng(1)
    mk = lambda s, e: (np.ldexp(rng.uniform(1, 2, s), e) * rng.choice([-1, 1], s)).astype(np.float32)
    A, B = mk(c.shapes()[0], ea), mk(c.shapes()[1], eb)
    C = np.zeros(c.shapes()[2], np.float32)
    ref, _ = _exact(A, B, C, 1.0, 0.0)
    err = lambda plan: np.sqrt(np.mean((run_gpu(c, A, B, C, prec=F32, plan=plan) - ref) ** 2))
    split, fp32 = err(_split(c, 0)), err(build_packed_plan(c.problem, F32, 2))
    print("2^%d 2^%d: split %.3e, FP32 MFMA %.3e (in 2^-149)" % (ea, eb, split * 2.0 ** 149, fp32 * 2.0 ** 149), flush=True)
    assert split <= fp32 + 2.0 ** -150


def _errors(k, dist, nonzero=None, tiles=SPLIT_RESIDENT):
    """2-norm errors of the split, tile by tile, and of the FP32 kernel; nonzero:
    that many values in a row of A, at random places."""
    c = _matmul(384, 320, k)
    A, B, C = inputs(c, k + 7 * (nonzero or 0), dist)
    if nonzero:
        rng = np.random.default_rng(k)
        A[np.argsort(rng.random(A.shape), axis=1) >= nonzero] = 0
    ref, _ = _exact(A, B, C, 1.0, 0.0)
    err = lambda plan: np.linalg.norm(run_gpu(c, A, B, C, prec=F32, plan=plan) - ref) / np.linalg.norm(ref)
    split, fp32 = [err(_split(c, t)) for t in tiles], err(build_packed_plan(c.problem, F32, 2))
    print("k %d %s %s: split %s, FP32 MFMA %.3e" % (k, dist, nonzero, ["%.3e" % e for e in split], fp32), flush=True)
    return split, fp32


@pytest.mark.parametrize("k", [32, 100, 2304])
@pytest.mark.parametrize("dist", ["uniform", "normal"])
def test_error_no_larger_than_the_fp32_kernels(k, dist):
    """Dense operands: one rounding in the larger sum for 16 k values, where the
    FP32 MFMA rounds once for two: from k = 32 on well under its error."""
    split, fp32 = _errors(k, dist)
    assert all(e <= 0.6 * fp32 for e in split)


@pytest.mark.parametrize("k", [32, 512])
@pytest.mark.parametrize("nonzero", [1, 2, 4, 8, 32])
@pytest.mark.parametrize("dist", ["uniform", "normal"])
def test_error_of_sums_of_few_products(k, nonzero, dist):
    """Rows of A with few nonzero values.  One product is rounded once either way;
    the split leaves out three part products of at most 2^-25 of it each, 0.41
    units of the rounding's 0.58 at most, so sqrt(1 + 0.41^2 / 3) = 1.03 times the
    error at one value (the left out products are uniform in their range), and no
    more than the FP32 MFMA's from two values on."""
    split, fp32 = _errors(k, dist, nonzero, (0, 7))
    assert all(e <= (1.05 if nonzero == 1 else 1.0) * fp32 for e in split)


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
