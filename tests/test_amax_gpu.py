"""The one-launch reduction behind the FP8 scales against torch: sizes around
its block, vector and grid edges, misaligned operands, special values, several
calls on one scratch array."""
import ctypes

import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nA, nB", [(1, 1), (3, 4), (5, 4095), (4096, 4097), (4096 * 511 + 7, 4096 * 512 + 5),
                                    (4096 * 700 + 3, 2)])
def test_amax_pair(nA, nB):
    import torch
    from tccg_amd.runtime import load_library
    lib = load_library()
    out = torch.zeros(lib.tccg_amax_pair_floats(), device="cuda")
    g = torch.Generator(device="cuda").manual_seed(nA)
    A = torch.randn(nA + 3, device="cuda", generator=g)
    B = torch.randn(nB + 3, device="cuda", generator=g)
    s = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    for off in range(4):                      # 4-byte steps off the 16-byte boundary
        for place in (0, -1):                 # the largest value first or last
            a, b = A[off:off + nA], B[3 - off:3 - off + nB]
            a[place], b[-1 - place] = -7.5 - off, 11.25 + off
            rc = lib.tccg_amax_pair_f32(a.data_ptr(), nA, b.data_ptr(), nB, out.data_ptr(), s)
            assert rc == 0
            torch.cuda.synchronize()
            assert out[0].item() == a.abs().max().item() and out[1].item() == b.abs().max().item()
    A[1] = float("nan")                       # as before: a NaN is passed over, an infinity is not
    B[1] = float("-inf")
    assert lib.tccg_amax_pair_f32(A.data_ptr(), nA, B.data_ptr(), nB, out.data_ptr(), s) == 0
    torch.cuda.synchronize()
    assert out[0].item() == torch.nan_to_num(A[:nA], nan=0.0).abs().max().item()
    assert out[1].item() == B[:nB].abs().max().item()
