"""Group sizes, K and N that do not come in whole chunks and tiles (mma.cuh:63-230, the reference's kernel, takes
any gs % 8 == 0 and zero-pads the edges): blocks and tiles at the edges where they can go wrong -- rows that end inside a
16-byte piece, a slice of 32 k, a chunk or a stage, groups that begin anywhere in a slice, scale arrays that end
inside a dword, matrices that end inside a tile of rows.

Outputs are held to 5e-4 of the FP64 oracle on sampled rows and columns (FP16 weights and outputs, FP32 sums: 2.1e-4 is
what these shapes measure; the reference's gate is 1e-3, tests/test_gpu.cu:184-193); hooked bytes are the oracle's."""
import numpy as np
import pytest
import torch

import orc
import w4amd
from devutil import DevPacked, DevPackedMx, bits, halves, ptr, to_dev

pytestmark = pytest.mark.gpu
TOL = 5e-4


def _check(fmt, M, N, K, gs, scale=None):
    c = w4amd.capi()
    seed = M + N + K + gs + fmt
    x = orc.normal_activations(M * K, seed)
    if fmt == 2:
        p = orc.quantize_mx(orc.outlier_weights(N, K, seed), N, K)
        dp, fn, w_ref = DevPackedMx(p), c.gemm_mma_mx, orc.dequant_all_mx(p)
    else:
        p = orc.quantize(orc.normal_weights(N * K, seed) * 0.02 + 0.01 * fmt, N, K, gs, fmt == 0)
        dp, fn, w_ref = DevPacked(p), c.gemm_mma, orc.dequant_all(p)
    x_d = to_dev(x)
    rng = np.random.default_rng(seed)
    ms = np.unique(np.concatenate([[0, M - 1], rng.choice(M, size=min(M, 20), replace=False)]))
    ns = np.unique(np.concatenate([np.arange(min(N, 40)), np.arange(max(0, N - 40), N), rng.choice(N, size=min(N, 80), replace=False)]))
    ref = orc.gemm_oracle(np.ascontiguousarray(x.reshape(M, K)[ms]), len(ms), K,
                          np.ascontiguousarray(w_ref.reshape(N, K)[ns]), len(ns))
    seen = []
    for hook in (False, True):
        out, w = halves(M * N + 64, 0x7E00), halves(N * K + 64, 0x7E00)
        fn(dp.view, ptr(x_d), ptr(out), M, 0, ptr(w) if hook else 0)
        got = bits(out)
        assert (got[M * N:] == 0x7E00).all(), "nothing is written behind the result"
        seen.append(got)
        got = np.ascontiguousarray(got[: M * N].reshape(M, N)[ms][:, ns]).view(np.float16)
        assert orc.rel_l2(got, ref) <= TOL, hook
        if hook:
            assert torch.equal(w[: N * K], to_dev(w_ref)) and bool((w[N * K:] == 0x7E00).all())
    assert np.array_equal(*seen), "the hook changes no byte of the result"
    return c.gemm_plan_for(fmt, M, N, K, gs)


# (plan, fmt, M, N, K, gs): tiles of 32 x 128 (4) to 128 x 256 (7) in every compiled form; K ends inside a chunk and, 264, 520 and
# 1032, inside a piece; gs = 40 .. 136 begin in any word; N * G odd (MXFP4: N * B % 4): the last scale is part of a dword
TILES = [(4, 0, 1100, 257, 2080, 24), (4, 0, 2049, 257, 1032, 8), (4, 0, 2049, 129, 1056, 72), (4, 0, 520, 257, 264, 40),
         (4, 1, 2049, 129, 2080, 24), (4, 1, 2049, 257, 1032, 24), (4, 1, 1100, 257, 1056, 40), (4, 1, 900, 777, 520, 40),
         (4, 2, 2049, 129, 1056, 32), (4, 2, 2049, 257, 1032, 32), (5, 0, 1300, 777, 2080, 24), (5, 0, 1300, 777, 264, 16),
         (5, 0, 1300, 777, 1056, 104), (5, 0, 900, 1034, 264, 48), (5, 1, 520, 2051, 2080, 24), (5, 1, 1300, 777, 264, 8),
         (5, 1, 1300, 777, 1056, 96), (5, 1, 1300, 777, 264, 40), (5, 2, 1700, 1034, 1056, 32), (5, 2, 1700, 1034, 1032, 32),
         (6, 0, 1100, 2051, 2080, 24), (6, 0, 1100, 2051, 264, 8), (6, 0, 1100, 2051, 1056, 104), (6, 0, 700, 3001, 264, 40),
         (6, 1, 900, 3001, 2080, 24), (6, 1, 1100, 2051, 264, 8), (6, 1, 700, 3001, 1056, 40), (6, 1, 700, 3001, 264, 96),
         (6, 2, 900, 2310, 1056, 32), (6, 2, 900, 2310, 264, 32), (7, 0, 1300, 3001, 1056, 1056), (7, 0, 1300, 3001, 264, 40),
         (7, 1, 2049, 2051, 1152, 40), (7, 1, 1300, 3001, 264, 128), (7, 2, 1700, 2310, 1056, 32), (7, 2, 1300, 3001, 264, 32),
         (4, 1, 130, 3001, 264, 40), (5, 2, 900, 1034, 1056, 32)]
# calls that tiles are behind in (us on tiles and on the kernels before): 8.1 and 7.5, 9.2 and 8.3, 6.0 and 5.8, 8.2 and 6.8
TILES_BEHIND = [(0, 2049, 257, 264, 8), (1, 900, 777, 264, 24), (2, 520, 257, 264, 32), (2, 900, 1034, 264, 32)]
BLOCKS = [(0, 5, 130, 4104, 8), (1, 9, 33, 3336, 24), (1, 17, 1034, 2056, 48), (0, 20, 15, 264, 40), (1, 33, 281, 1000, 16), (0, 50, 513, 5176, 72),
          (1, 64, 3, 1032, 1032), (1, 40, 2063, 4104, 8), (0, 100, 129, 2080, 128), (1, 130, 40, 1384, 48), (2, 17, 281, 1000, 32), (2, 50, 7, 3336, 32),
          (2, 130, 1001, 2072, 32), (1, 100, 2064, 1152, 48), (0, 333, 4080, 4096, 48), (1, 64, 3000, 2048, 96), (0, 120, 1477, 2304, 128),
          (1, 48, 1477, 4096, 32),
          # parameters that LDS holds a window of units at a time: three of one tile of W, two and three of two; the
          # last window shorter, waves without a unit in it
          (0, 17, 515, 20480, 8), (1, 70, 2050, 11024, 8), (0, 100, 2064, 12304, 8), (1, 33, 1034, 20496, 16),
          # the general decode kernel would take three rounds, its LDS holds one tile's parameters
          (1, 61, 11008, 4096, 8)]


@pytest.mark.parametrize("plan,fmt,M,N,K,gs", TILES)
def test_tiles_of_any_group(plan, fmt, M, N, K, gs):
    assert _check(fmt, M, N, K, gs) == plan


@pytest.mark.parametrize("fmt,M,N,K,gs", TILES_BEHIND)
def test_calls_that_tiles_are_behind_in(fmt, M, N, K, gs):
    assert _check(fmt, M, N, K, gs) == 0


@pytest.mark.parametrize("fmt,M,N,K,gs", BLOCKS)
def test_blocks_of_any_group(fmt, M, N, K, gs):
    assert _check(fmt, M, N, K, gs) >= 10


@pytest.mark.parametrize("M,N,K", [(300, 1302, 1160), (50, 282, 2088), (1300, 2050, 1048)])
@pytest.mark.parametrize("gs", [8, 48, 0])
def test_ends_of_rows_bring_no_infinity(M, N, K, gs):
    """The codes that stand in for a row's end are other groups', here with scales that overflow FP16, and the activations
    that the last stage shares with the one before it are infinite in one row: results are infinite where the oracle's
    are, NaN nowhere else."""
    mx = gs == 0
    rng = np.random.default_rng(M + K + gs)
    G = (K + 31) // 32 if mx else (K + gs - 1) // gs
    codes = rng.integers(0, 16, (N, K))
    codes[:, (G - 1) * (gs or 32):] = 2 if mx else 9  # 1.0
    words = (codes.reshape(N, K // 8, 8).astype(np.uint64) << (4 * np.arange(8, dtype=np.uint64))).sum(-1).astype(np.uint32)
    c = w4amd.capi()
    x = orc.normal_activations(M * K, 3).view(np.float16).reshape(M, K).copy()
    x[2, K - 100] = np.inf  # in the stage before the last as well
    if mx:
        p = orc.quantize_mx(np.ones(N * K), N, K)
        s = np.full((N, G), 127 - 6, np.uint8)
        s[:, -1] = 127 + 14
        dp, fn = (lambda: DevPackedMx(p)), c.gemm_mma_mx
    else:
        p = orc.quantize(np.ones(N * K), N, K, gs, True)
        s = np.full((N, G), 0.01, np.float16)
        s[:, -1] = 60000
        s = s.view(np.uint16)
        dp, fn = (lambda: DevPacked(p)), c.gemm_mma
    p.q[:], p.scales[:] = words.ravel(), s.ravel()
    x[:, (G - 1) * (gs or 32):] *= np.float16(2.0 ** -12)
    w = (orc.dequant_all_mx(p) if mx else orc.dequant_all(p)).view(np.float16).reshape(N, K).astype(np.float64)
    d, out = dp(), halves(M * N)
    fn(d.view, ptr(to_dev(x.view(np.uint16).ravel())), ptr(out), M)
    got = bits(out).view(np.float16).reshape(M, N).astype(np.float64)
    rows = np.array([0, 1, 3, M - 1])
    with np.errstate(invalid="ignore"):
        ref = x[rows].astype(np.float64) @ w.T
        bad = x[2].astype(np.float64)[None] @ w.T
    # an output is finite where the oracle's stays below the largest half by more than 2^-10 of the sum of magnitudes (FP32 sums
    # of K < 2^13 products are off by less than 2^-11 of it)
    sure = np.abs(ref) < 65504 - 2.0 ** -10 * (np.abs(x[rows].astype(np.float64)) @ np.abs(w.T))
    assert sure.mean() > 0.9 and not np.isnan(got[rows]).any() and np.isfinite(got[rows][sure]).all()
    assert np.isfinite(ref).any() and np.isfinite(got[rows]).sum() >= np.isfinite(ref).sum() * 0.99
    ok = np.isfinite(ref) & np.isfinite(got[rows])
    assert np.linalg.norm((got[rows] - ref)[ok]) <= 1e-3 * np.linalg.norm(ref[ok])
    assert np.array_equal(np.isnan(got[2]), np.isnan(bad[0])) and np.array_equal(np.isinf(got[2]), np.isinf(bad[0]))


@pytest.mark.parametrize("M,N,K", [(136, 1639, 1152), (500, 2050, 384), (129, 2048, 128), (1100, 1024, 1024), (70, 2306, 1280)])
def test_thin_grids_of_32_groups_with_zero_points(M, N, K):
    """gs = 32 with zero-points on the two smallest tiles (one stage, an odd number of them, ragged rows): the hooked kernel
    splits its sum over K at the same stage, so both calls return the same bytes."""
    c = w4amd.capi()
    assert _check(1, M, N, K, 32) == 0
    p = orc.quantize(orc.normal_weights(N * K, 7) * 0.02 + 0.01, N, K, 32, False)
    dp, x_d = DevPacked(p), to_dev(orc.normal_activations(M * K, 8))
    plain, hooked, w = halves(M * N), halves(M * N), halves(N * K)
    c.gemm_mma(dp.view, ptr(x_d), ptr(plain), M)
    c.gemm_mma(dp.view, ptr(x_d), ptr(hooked), M, 0, ptr(w))
    assert torch.equal(plain, hooked)


@pytest.mark.parametrize("M,N,K,gs,sym", [(1134, 736, 576, 128, False), (222, 9776, 576, 256, True), (180, 11648, 1504, 128, True),
                                          (128, 2064, 1504, 128, True), (559, 5728, 1056, 128, False)])
def test_groups_of_whole_chunks_keep_their_scales_in_fp32(M, N, K, gs, sym):
    """Groups of whole chunks, K no multiple of one: the scale belongs to FP32 sums and no weight is rounded.  Distance from the
    FP64 product of codes and scales: an output rounded to FP16 alone is 2^-10 / sqrt(12) sqrt(E m^-2) = 2.1e-4 off (m: significands
    spread over their logarithm), rounded weights add 1.7e-4 to it in squares (2.7e-4)."""
    c = w4amd.capi()
    p = orc.quantize(orc.normal_weights(N * K, M) * 0.02 + (0 if sym else 0.01), N, K, gs, sym)
    dp, x, out = DevPacked(p), orc.normal_activations(M * K, N), halves(M * N)
    assert c.gemm_plan_for(0 if sym else 1, M, N, K, gs) >= 10
    c.gemm_mma(dp.view, ptr(to_dev(x)), ptr(out), M)
    ns = np.random.default_rng(K).choice(N, 256, replace=False)
    code = (p.q.reshape(N, K // 8)[ns][:, :, None] >> (4 * np.arange(8, dtype=np.uint32))) & 15
    group = np.arange(K) // gs
    zero = np.full((256, K), 8.0)
    if not sym:
        zero = ((p.zeros.reshape(N, -1)[ns][:, group // 8] >> (4 * (group % 8)).astype(np.uint32)) & 15).astype(np.float64)
    w = (code.reshape(256, K) - zero) * p.scales.view(np.float16).reshape(N, -1)[ns][:, group].astype(np.float64)
    ref = x.view(np.float16).reshape(M, K).astype(np.float64) @ w.T
    assert orc.rel_l2(np.ascontiguousarray(bits(out).reshape(M, N)[:, ns]).view(np.float16), ref) <= 2.4e-4


def test_blocks_along_more_rows_of_w_than_one_grid_dimension_has():
    """N = 17 million: more blocks of W (eight a row of the grid) than 65535, the grid's second dimension; columns around its end."""
    c = w4amd.capi()
    M, N, K = 17, 17_000_007, 1032
    assert c.gemm_plan_for(0, M, N, K, K) in (11, 21, 22, 24) and N > 65535 * 8 * 32
    q = torch.empty(N, K // 8, dtype=torch.int32, device="cuda")
    q.random_(-2 ** 31, 2 ** 31 - 1, generator=torch.Generator(device="cuda").manual_seed(5))
    s = (torch.rand(N, 1, device="cuda") * 0.01 + 0.01).half()
    x, out = torch.randn(M, K, device="cuda").half(), torch.full((M, N), float("nan"), dtype=torch.float16, device="cuda")
    c.gemm_mma(c.packed_view(N, K, K, 1, True, ptr(q), ptr(s)), ptr(x), ptr(out), M)
    for n in (0, 65535 * 8 * 16, 65535 * 8 * 32, N):
        ns = slice(max(0, n - 200), min(N, n + 200))
        code = (q[ns][:, :, None] >> (4 * torch.arange(8, device="cuda"))) & 15
        w = ((code.reshape(-1, K) - 8) * s[ns].float()).half().double()
        ref = (x.double() @ w.T).cpu().numpy()
        assert orc.rel_l2(out[:, ns].contiguous().cpu().numpy(), ref) <= TOL, n
    assert not bool(torch.isnan(out).any())


# Calls that the kernels before are ahead in, and calls beside them in which blocks or tiles are (us then and now): the times of both
# sides depend on whole 16-byte pieces of codes, on steps that the stream kernel's ring rounds up, on outputs stored one by one
PLAN = [((1, 3991, 1551, 2048, 16), False), ((1, 3991, 1551, 2056, 16), True),    # 52 and 72
        ((0, 5, 15272, 1408, 128), False), ((0, 5, 15272, 4104, 128), True),      # 6.6 and 9.5
        ((1, 2964, 304, 352, 64), False), ((1, 2964, 304, 1056, 64), True),       # 5.7 and 8.4
        ((2, 30, 16320, 352, 32), False), ((2, 30, 16320, 1056, 32), True),       # 4.5 and 6.1
        ((1, 9, 8778, 1792, 1792), False), ((1, 9, 8778, 4096, 4096), True),      # 7.8 and 9.8
        ((1, 3052, 2271, 256, 96), False), ((1, 3052, 2272, 264, 96), True),      # 20.6 and 25.1
        # small groups with zero-points on the stream kernel: 11.1 and 19.9
        ((1, 53, 9712, 1024, 8), True), ((1, 20, 13824, 1024, 16), True),           # 9.5 and 18.8
        # gs = 32 with zero-points, blocks against its two smallest tiles (plan 0): 6.0 and 7.1, 7.4 and 8.0
        ((1, 68, 5712, 384, 32), False), ((1, 68, 2736, 384, 32), True), ((1, 66, 6464, 640, 32), False), ((1, 66, 4704, 640, 32), True)]


@pytest.mark.parametrize("call,ahead", PLAN)
def test_blocks_and_tiles_are_planned_where_they_are_ahead(call, ahead):
    assert (w4amd.capi().gemm_plan_for(*call) >= 4) == ahead
