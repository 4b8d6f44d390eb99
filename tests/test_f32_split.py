"""Plans that run FP32 contractions on the BF16 MFMAs (split_plans), host side:
which values the three parts hold, which contractions get such a plan, and the
workspace with its guard words."""
import ctypes

import numpy as np
import pytest

from oracle.precision_ref import split_bf16_parts
from tccg_amd import Contraction, build
from tccg_amd.plan import (BF16X3, F32, F64, PACKED_TAIL_BYTES, PACKED_TILES, SPLIT_MIN_K, build_packed_plan, call_plan,
                           default_plan, split_plans)


SCALE = 23   # kSplitScale of gett_core.hpp: the parts are those of x 2^23


def limit(Kp: int) -> int:
    """h of split_limit() in gett_pack.hpp: |x| < 2^h is held."""
    return (81 - (Kp - 1).bit_length()) // 2


@pytest.mark.parametrize("e", [-149, -148, -140, -127, -126, -125, -100, -1, 0, 1, 33, 37])
def test_parts_hold_every_accepted_value(e):
    """Every mantissa pattern class at the edges of the accepted exponents,
    subnormals among them: the three parts add up to the scaled value exactly, in
    FP32 from the smallest up, and each is zero or a normal BF16 number."""
    rng = np.random.default_rng(e + 200)
    man = np.concatenate([np.arange(64), (1 << 23) - 1 - np.arange(64), rng.integers(0, 1 << 23, 20000),
                          (rng.integers(0, 128, 500) << 16) | 0x8000, (rng.integers(0, 1 << 15, 500) << 8) | 0x80])
    x = np.concatenate([s * np.ldexp(1.0 + man / 2.0 ** 23, e) for s in (1, -1)]).astype(np.float32)
    xs = x * np.float32(2.0 ** SCALE)
    assert np.array_equal(xs.astype(np.float64), x.astype(np.float64) * 2.0 ** SCALE)
    p0, p1, p2 = (p.astype(np.float32) for p in split_bf16_parts(xs))
    assert np.array_equal(p0 + (p1 + p2), xs)
    for p in (p0, p1, p2):
        assert np.all((p == 0) | (np.abs(p) >= 2.0 ** -126))


@pytest.mark.parametrize("Kp", [32, 64, 96, 2304, 4096, 4128, 1 << 20])
def test_held_values_cannot_overflow(Kp):
    """Kp products of the largest first parts (2^(h + 23) each) stay under 2^127,
    and the limit is the largest that a sum of Kp products allows in this form."""
    h = limit(Kp)
    assert Kp * 2.0 ** (2 * (h + SCALE)) <= 2.0 ** 127
    assert 2.0 ** (Kp - 1).bit_length() * 2.0 ** (2 * (h + 1 + SCALE)) > 2.0 ** 127
    assert h >= 27


def _matmul(m, n, k):
    return Contraction.from_labels(["m", "n"], ["k", "m"], ["n", "k"], {"m": m, "n": n, "k": k})


def test_which_contractions_get_a_split_plan():
    big = _matmul(2048, 2048, 1024)
    assert all(p.guard and p.packed and p.prec == BF16X3 and p.walk in (0, 5) and p.ksplit == 1
               for p in split_plans(big.problem))
    assert call_plan(big.problem, F32).guard
    # other precisions and the plans of the code generators are untouched
    assert not call_plan(big.problem, BF16X3).guard and not call_plan(big.problem, F64).guard
    assert not default_plan(big.problem, F32).guard and big.plan("f32").prec == F32
    assert split_plans(_matmul(512, 512, SPLIT_MIN_K).problem)
    assert not split_plans(_matmul(512, 512, SPLIT_MIN_K - 1).problem)


@pytest.mark.parametrize("m, n, k", [(64, 64, 32), (65, 300, 33), (700, 129, 500)])
def test_workspace_holds_the_guard_words(m, n, k):
    path = build.library_path()
    if not path.exists():
        pytest.skip("library not built")
    from tccg_amd.runtime import _CPlan, load_library
    lib = load_library()
    pb = _matmul(m, n, k).problem
    for t, kw in ((0, {}), (4, {}), (5, dict(stream_k=1)), (6, dict(persistent=True))):
        plain = build_packed_plan(pb, BF16X3, t, **kw)
        p = build_packed_plan(pb, BF16X3, t, guard=True, **kw)
        cp = _CPlan()
        cp.Mp, cp.Np, cp.Kp, cp.tile, cp.walk, cp.grid = p.Mp, p.Np, p.Kp, p.tile, p.walk, p.grid
        assert lib.tccg_f32_split_workspace_bytes(ctypes.byref(cp)) == p.workspace_bytes()
        off = lib.tccg_f32_split_clear_offset(ctypes.byref(cp))
        words = (p.Mp // 64 + p.Np // 64) * (p.Kp // 32)
        # after every byte of the split-BF16 plan's, before the prefetch's tail
        assert off % 256 == 0 and off >= plain.workspace_bytes() - PACKED_TAIL_BYTES
        assert off + 256 + 4 * words <= p.workspace_bytes() - PACKED_TAIL_BYTES
    for t in (7, 8):
        p = build_packed_plan(pb, BF16X3, t, guard=True)
        assert (p.BM, p.BN, p.BK) == PACKED_TILES[BF16X3][t] and p.Mp % p.BM == p.Np % p.BN == 0
        cp = _CPlan()
        cp.Mp, cp.Np, cp.Kp, cp.tile, cp.walk, cp.grid = p.Mp, p.Np, p.Kp, p.tile, p.walk, p.grid
        assert lib.tccg_f32_split_workspace_bytes(ctypes.byref(cp)) == p.workspace_bytes()


def test_operands_beyond_the_packed_limit_keep_the_fp32_plan():
    """The packed planes address 2^32 - 1 elements: a contraction whose FP32
    planes fit but whose three BF16 parts do not keeps its FP32 plan."""
    from tccg_amd import plan as P
    pb = _matmul(40000, 128, 40000).problem
    assert 40000 * 40000 < 2 ** 32 - 1 < 3 * 40000 * 40000
    assert not P.split_fits(build_packed_plan(pb, BF16X3, 0))
    assert P.split_fits(build_packed_plan(_matmul(20000, 128, 20000).problem, BF16X3, 0))


def test_entry_rejects_what_it_cannot_run():
    path = build.library_path()
    if not path.exists():
        pytest.skip("library not built")
    from tccg_amd.runtime import _CPlan, load_library
    lib = load_library()
    assert lib.tccg_gett_f32_split(None, None, None, 1.0, 0.0, None, None, 0, 0, None) != 0
    p = build_packed_plan(_matmul(512, 512, 512).problem, BF16X3, 0)
    cp = _CPlan()
    cp.Mp, cp.Np, cp.Kp, cp.tile = p.Mp, p.Np, p.Kp, p.tile
    one = ctypes.c_void_p(256)   # never dereferenced: every call below is rejected before a launch
    for f in ("offAm", "offAk", "offBn", "offBk", "offCm", "offCn"):
        setattr(cp, f, 256)
    need = lib.tccg_f32_split_workspace_bytes(ctypes.byref(cp))
    assert lib.tccg_gett_f32_split(one, one, one, 1.0, 0.0, ctypes.byref(cp), one, need - 1, 0, None) != 0
    assert b"workspace too small" in lib.tccg_last_error()
    cp.ksplit = 2
    assert lib.tccg_gett_f32_split(one, one, one, 1.0, 0.0, ctypes.byref(cp), one, 1 << 40, 0, None) != 0
    assert b"without ksplit" in lib.tccg_last_error()


@pytest.mark.parametrize("m, n, k", [(221, 3124, 2401), (930, 840, 4002), (1239, 1936, 928), (5184, 5184, 2304),
                                     (128, 128, 32), (64, 64, 20000), (300, 300, 511)])
def test_calls_do_not_lengthen_the_summation_chains(m, n, k):
    """FP32 calls add up at most 1.3 times the k values one after the other
    that stream-k over 128x128 tiles would (512 where that is less)."""
    from tccg_amd.plan import _chain
    pb = Contraction.from_labels(["m", "n"], ["k", "m"], ["n", "k"], {"m": m, "n": n, "k": k}).problem
    tiles = -(-m // 128) * -(-n // 128)
    split = split_plans(pb)
    if not split:                             # no split plan cuts k finely enough
        assert call_plan(pb, F32).describe() == default_plan(pb, F32).describe()
    for p in split and [call_plan(pb, F32)] + split:
        assert _chain(p) <= max(512, 1.3 * k * min(1.0, tiles / 256)), p.describe()


# (m, n, k) of a product and the full-size roundings of the plans that were chosen
# for it in FP32, FP64 and split-BF16 when the launch estimate was fitted to larger
# tiles and stream-k (split-BF16: six per 16 k values, in one sum).
ROUNDINGS = [
    (930, 840, 4002, 446, 226, 336),
    (1152, 640, 896, 449, 46, 337),
    (2414, 598, 1420, 271, 137, 204),
    (1840, 1460, 480, 241, 87, 181),
    (930, 3264, 2296, 387, 470, 704),
    (2296, 930, 3264, 388, 461, 691),
    (221, 3124, 2401, 244, 125, 185),
    (247, 840, 4200, 2101, 77, 1576),
    (4200, 247, 840, 421, 60, 316),
    (480, 1496, 1554, 778, 80, 584),
    (2150, 494, 2688, 361, 183, 272),
    (2520, 352, 1536, 769, 95, 140),
    (3192, 275, 2691, 403, 204, 303),
    (1976, 558, 986, 494, 82, 205),
    (3332, 1725, 1200, 387, 301, 451),
    (4980, 1344, 2679, 958, 671, 719),
    (3149, 2076, 3344, 1230, 837, 923),
    (1320, 800, 190, 96, 28, 73),
    (726, 840, 431, 217, 40, 163),
    (312, 1848, 672, 337, 52, 253),
    (64, 64, 20000, 10001, 1254, 7501),
    (128, 128, 32, 17, 9, 13),
    (300, 300, 511, 257, 36, 193),
    (5184, 5184, 2304, 1153, 577, 865),
    (99, 810, 1450, 726, 48, 545),
    (2065, 493, 3654, 493, 249, 371),
    (583, 1788, 3273, 455, 230, 342),
    (48, 48, 48, 25, 13, 19),
    (480, 282, 269, 136, 38, 102),
    (3392, 1815, 3087, 1093, 773, 1159),
    (175, 1763, 358, 180, 50, 135),
]


@pytest.mark.parametrize("m, n, k, f32, f64, bf16x3", ROUNDINGS)
def test_no_plan_rounds_more_often_than_those_chosen_before(m, n, k, f32, f64, bf16x3):
    """The plans of calls and of the code generators: the error grows with the root
    of the count, 3 % of it is the allowance for padded k-steps."""
    from tccg_amd.plan import _roundings
    pb = _matmul(m, n, k).problem
    for prec, before in ((F32, f32), (F64, f64), (BF16X3, bf16x3)):
        for plan in (default_plan(pb, prec), call_plan(pb, prec)):
            assert _roundings(plan) <= 1.03 ** 2 * before, plan.describe()


def test_roundings_of_a_plan():
    from tccg_amd.plan import _roundings
    pb = _matmul(256, 256, 1024).problem
    assert _roundings(build_packed_plan(pb, F32, 0)) == 1024 / 2 + 1
    assert _roundings(build_packed_plan(pb, F32, 0, ksplit=4)) == 256 / 2 + 4
    assert _roundings(build_packed_plan(pb, F64, 0, stream_k=1)) == 1024 * 4 / 256 / 4 + 64   # 4 tiles on 256
    assert _roundings(build_packed_plan(pb, BF16X3, 0)) == 1024 / 16 + 1 + 1


@pytest.mark.parametrize("n, min_k", [(8, 8), (40, 8), (3, 1)])
def test_group_candidates_are_different_launches(n, min_k):
    """Each (tile, order) choice of a batch is a launch of its own, whether the
    batch runs on the BF16 MFMAs or (a k range under four) on the FP32 ones."""
    from tccg_amd.batch import group_candidates, group_plans, random_batch
    cs = random_batch(n, seed=n)
    if min_k < 4:
        cs.append(_matmul(40, 30, min_k))
    launches = [((group_plans(cs, t)[0].prec, group_plans(cs, t)[0].tile), order) for t, order, _ in group_candidates(cs)]
    assert len(set(launches)) == len(launches) >= 8
    every = {(p.prec, p.tile) for t in range(len(PACKED_TILES[F32])) for p in group_plans(cs, t)}
    assert {l for l, _ in launches} == every   # and no launch is left out
