"""-m gpu: the few-row GEMM (csrc/kernels_gemm_skinny.hip), which launch_gemm takes by itself for these shapes (where it does not, the tiled kernels
are held to the same bounds: the cases say so), against the oracle chain."""
import pytest
import torch

from aha_amd import _lib
from oracle import qwen3 as oq
from tests.test_ops_gpu import NM, assert_close_ulps, rnd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [1, 8, 9, 16, 17, 32, 33, 64])
@pytest.mark.parametrize("N,K", [
    (8, 768),        # one eight-row group, as many k chunks per wave as ring stages; 33 and 64 rows: the tiles (below 2 MB)
    (1264, 832),     # N ends inside a block of 16, 24, 32 and 48 rows; an uneven share of chunks per wave
    (6144, 768),     # 24 rows per block: half a fragment unused
    (12320, 832),    # 32 rows per block in two rounds; 64 rows: the tiles
    (40, 4160),      # many chunks; 33 and 64 rows: the tiles
])
def test_few_rows_every_row_count_and_block_width(gpu, M, N, K):
    """One f32 sum per element, rounded once per op as in the tiled kernels: a sum next to a rounding boundary moves one op's result by one ulp, so
    1 ulp for the plain product, 2 behind bias and residual, 3 behind the GELU (whose hardware exp2 adds one; no share of equal bits is asked for:
    far in its tail the results are below 2^-8 of the rms and carry no comparable bits).  The rows behind M of the output stay untouched."""
    from aha_amd import ops, _lib
    from aha_amd._lib import check, lib
    A, W, b, r = rnd((M, K), 51), rnd((N, K), 52, 0.05), rnd((N,), 53, 0.5), rnd((M, N), 54)
    Ad, Wd, bd, rd = (t.to(gpu) for t in (A, W, b, r))
    out = torch.full((M + 3, N), 7.0, dtype=torch.bfloat16, device=gpu)
    check(lib().aha_hip_gemm(Ad.data_ptr(), Wd.data_ptr(), out.data_ptr(), M, N, K, K, K, N, None, None, _lib.ACT_NONE, torch.cuda.current_stream().cuda_stream))
    assert_close_ulps(out[:M], NM.linear(A.float(), W.float()), 1, None, "plain")
    assert (out[M:] == 7.0).all()
    assert torch.equal(ops.gemm(Ad, Wd), out[:M])
    full = ops.gemm(Ad, Wd, bd, rd, _lib.ACT_NONE)
    assert_close_ulps(full, NM.r(r.float() + NM.linear(A.float(), W.float(), b.float())), 2, None, "bias + residual")
    gelu = NM.r(torch.nn.functional.gelu(NM.linear(A.float(), W.float(), b.float()), approximate="tanh"))
    assert_close_ulps(ops.gemm(Ad, Wd, bd, None, _lib.ACT_GELU_TANH), gelu, 3, None, "bias + gelu")


@pytest.mark.parametrize("M", [1, 8, 13, 31, 64])
@pytest.mark.parametrize("I,K", [(16, 768), (1008, 832), (3072, 1024), (12288, 768)])
def test_few_rows_gate_up_pairs(gpu, M, I, K):
    """Gate and up rows in groups of eight per block, the product in the epilogue (interleaved layout of the model loader).  64 rows of the first and the
    last shape: the tiles."""
    from aha_amd import ops, _lib
    A, Wg, Wu = rnd((M, K), 61), rnd((I, K), 62, 0.05), rnd((I, K), 63, 0.05)
    ref = NM.r(NM.r(oq.silu(NM.linear(A.float(), Wg.float()))) * NM.linear(A.float(), Wu.float()))
    got = ops.gemm(A.to(gpu), ops.interleave_gate_up(Wg, Wu).to(gpu), None, None, _lib.ACT_SILU_MUL_PAIRS)
    assert_close_ulps(got, ref, 3, None, "gate * up")


@pytest.mark.parametrize("M", [65, 128, 129, 256])
@pytest.mark.parametrize("N,K,pairs", [(1024, 2048, False), (2056, 1088, False), (2720, 832, True)])
def test_row_tiles(gpu, M, N, K, pairs):
    """More than 64 rows in tiles of 64: the first and last of a tile, the last row count that comes here; bounds as above."""
    from aha_amd import ops, _lib
    A, W = rnd((M, K), 71), rnd((N, K), 72, 0.05)
    if pairs:
        ref = NM.r(NM.r(oq.silu(NM.linear(A.float(), W[:N // 2].float()))) * NM.linear(A.float(), W[N // 2:].float()))
        assert_close_ulps(ops.gemm(A.to(gpu), ops.interleave_gate_up(W[:N // 2], W[N // 2:]).to(gpu), None, None, _lib.ACT_SILU_MUL_PAIRS), ref, 3, None, "gate * up")
        return
    b, r = rnd((N,), 73, 0.5), rnd((M, N), 74)
    assert_close_ulps(ops.gemm(A.to(gpu), W.to(gpu)), NM.linear(A.float(), W.float()), 1, None, "plain")
    full = ops.gemm(A.to(gpu), W.to(gpu), b.to(gpu), r.to(gpu), _lib.ACT_NONE)
    assert_close_ulps(full, NM.r(r.float() + NM.linear(A.float(), W.float(), b.float())), 2, None, "bias + residual")


def rows_per_block(M, N, K, act=0):
    return _lib.lib().aha_hip_debug_few_rows_gemm(M, N, K, act, 0, 0, 1 << 30)   # 0: the tiled kernels


@pytest.mark.parametrize("N,K,width,M", [(N, K, w, M) for N, K, w, most in [(1272, 832, 16, 64), (5000, 832, 24, 64), (12312, 768, 32, 33), (12280, 832, 48, 64)]
                                         for M in (1, 8, 9, 16, 17, 32, 33, 64) if M <= most])
def test_block_width_with_pitches(gpu, N, K, width, M):
    """Every width of a block (asked for, so that a change of the cost model does not empty this test), N ending inside the last one, with rows of A, W,
    bias + residual and C that lie further apart than they are long; what lies between C's rows and behind them stays untouched.  1 ulp for the plain
    product, 2 behind bias and residual, as above."""
    from aha_amd._lib import check, lib
    assert rows_per_block(M, N, K) == width and N % width != 0
    lda, ldw, ldc = K + 8, K + 24, N + 12
    A, W, b, r = rnd((M, lda), 81), rnd((N, ldw), 82, 0.05), rnd((N,), 83, 0.5), rnd((M, ldc), 84)
    Ad, Wd, bd, rd = (t.to(gpu) for t in (A, W, b, r))
    ref = NM.linear(A[:, :K].float(), W[:, :K].float())
    st = torch.cuda.current_stream().cuda_stream
    for bias, res, want, ulps in ((None, None, ref, 1),
                                  (bd, rd, NM.r(r[:, :N].float() + NM.linear(A[:, :K].float(), W[:, :K].float(), b.float())), 2)):
        out = torch.full((M + 2, ldc), 7.0, dtype=torch.bfloat16, device=gpu)
        check(lib().aha_hip_gemm(Ad.data_ptr(), Wd.data_ptr(), out.data_ptr(), M, N, K, lda, ldw, ldc, bias.data_ptr() if bias is not None else None,
                                 res.data_ptr() if res is not None else None, _lib.ACT_NONE, st))
        assert_close_ulps(out[:M, :N], want, ulps, None, "pitched")
        assert (out[:M, N:] == 7.0).all() and (out[M:] == 7.0).all()


@pytest.mark.parametrize("M", [129, 192, 193, 255])
@pytest.mark.parametrize("act", ["plain", "bias + residual", "gate * up"])
def test_one_row_of_tall_tiles(gpu, M, act):
    """129 to 255 rows of a long W on the automatic plan: 256 x 128 tiles, the only row of them partly filled, the last column of them too; rows of A and
    W further apart than they are long.  Bounds as above."""
    import ctypes
    from aha_amd._lib import check, lib
    pairs = act == "gate * up"
    N, K, code = (16544 if pairs else 16520), 640, _lib.ACT_SILU_MUL_PAIRS if pairs else _lib.ACT_NONE
    plan = (ctypes.c_int32 * 3)()
    check(lib().aha_hip_debug_plan_gemm(M, N, K, code, act == "bias + residual", act == "bias + residual", 1 << 30, plan))
    assert tuple(plan) == (2128, 1, 0) and rows_per_block(M, N, K, code) == 0
    from aha_amd import ops
    A, W = rnd((M, K + 8), 91), rnd((N, K), 92, 0.05)
    Ad = A.to(gpu)
    ref = NM.linear(A[:, :K].float(), W.float())
    st = torch.cuda.current_stream().cuda_stream
    Wd = (ops.interleave_gate_up(W[:N // 2], W[N // 2:]) if pairs else W).to(gpu)
    No = N // 2 if pairs else N
    b, r = rnd((N,), 93, 0.5), rnd((M, No), 94)
    bd, rd = b.to(gpu), r.to(gpu)
    out = torch.full((M + 2, No), 7.0, dtype=torch.bfloat16, device=gpu)
    res = act == "bias + residual"
    check(lib().aha_hip_gemm(Ad.data_ptr(), Wd.data_ptr(), out.data_ptr(), M, N, K, K + 8, K, No, bd.data_ptr() if res else None, rd.data_ptr() if res else None, code, st))
    if pairs:
        ref = NM.r(NM.r(oq.silu(ref[:, :N // 2])) * ref[:, N // 2:])
    elif res:
        ref = NM.r(r.float() + NM.linear(A[:, :K].float(), W.float(), b.float()))
    assert_close_ulps(out[:M], ref, {"plain": 1, "bias + residual": 2, "gate * up": 3}[act], None, act)
    assert (out[M:] == 7.0).all()
