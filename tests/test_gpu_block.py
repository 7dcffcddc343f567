"""The block kernel of middle M (9 to a few hundred rows, at long K from 3 on; mma.cuh:234-260 is the reference's
dispatch for these shapes): every block shape at the edges where it can go wrong -- rows of x and of
W that end inside a block or a tile, K that ends inside a unit of 256 or a chunk of 128, waves
without a unit, group sizes from 32 to a whole row.

A hooked call takes the same kernel, so its output is compared byte for byte with the unhooked one;
its weights are the oracle's bytes; the output is within 1e-3 of the FP64 oracle (the reference's
gate, tests/test_gpu.cu:184-193)."""
import numpy as np
import pytest
import torch

import orc
import w4amd
from devutil import DevPacked, DevPackedMx, bits, halves, ptr, to_dev

pytestmark = pytest.mark.gpu
TOL = 1e-3


def _check(fn, view, w_ref, x, M, N, K, seed):
    x_d, w_ref_d = to_dev(x), to_dev(w_ref)
    # a guard row past the result and past the weights: nothing is written behind them
    c_h, c_u, w_d = halves(M * N + N, 0x7E00), halves(M * N + N, 0x7E00), halves(N * K + 64, 0x7E00)
    fn(view, ptr(x_d), ptr(c_h), M, 0, ptr(w_d))
    fn(view, ptr(x_d), ptr(c_u), M, 0, 0)
    assert torch.equal(w_d[: N * K], w_ref_d), "w_out bitwise"
    assert bool((w_d[N * K:] == 0x7E00).all()) and bool((c_u[M * N:] == 0x7E00).all())
    assert torch.equal(c_h, c_u), "hooked and unhooked calls are one kernel"
    rng = np.random.default_rng(seed)
    ms = np.unique(np.concatenate([[0, min(15, M - 1), min(16, M - 1), M - 1], rng.choice(M, size=min(M, 24), replace=False)]))
    ns = np.unique(np.concatenate([[0, 15, N - 1], rng.choice(N, size=min(N, 160), replace=False)]))
    ref = orc.gemm_oracle(np.ascontiguousarray(x.reshape(M, K)[ms]), len(ms), K,
                          np.ascontiguousarray(w_ref.reshape(N, K)[ns]), len(ns))
    got = np.ascontiguousarray(bits(c_u)[: M * N].reshape(M, N)[ms][:, ns]).view(np.float16)
    assert orc.rel_l2(got, ref) <= TOL


# (M, N, K): rows of x and of W that end inside a block or a tile, short and long K.  (test_every_block names the
# block; those marked * are another kernel's for most group sizes, and hooked and unhooked calls agree there too.)
SHAPES = [
    (3, 528, 4352),     # * long-K kernel
    (16, 4096, 2304),   # * long-K kernel
    (9, 8208, 4384),    # 64 x 16 blocks at the resident kernel's widths, ragged N and K
    (17, 272, 256),     # one unit: seven waves have none; N ends inside a block
    (33, 528, 4096),    # one tile of W a workgroup, two tiles of x, the third row of tiles one row high
    (48, 2064, 2336),   # K ends inside a chunk, in a unit of its own
    (100, 4096, 1152),  # 32 x 64 blocks; half a unit at the end
    (128, 6144, 512),   # * direct-to-LDS tiles; gs = 32 with zero-points: 48 x 64 blocks
    (96, 8208, 1024),   # * the same; 64 x 96 blocks
    (190, 4112, 2304),  # * the same; 64 x 64
    (150, 11008, 2048), # * direct-to-LDS tiles (two rounds of blocks)
    (333, 4080, 2176),  # * direct-to-LDS tiles
]


@pytest.mark.parametrize("M,N,K", SHAPES)
@pytest.mark.parametrize("gs,sym", [(128, True), (64, False), (32, True), (32, False), (0, False)])
def test_w4_block(M, N, K, gs, sym):
    if gs == 0:
        gs = K  # one group per row
    c = w4amd.capi()
    seed = M + N + K + gs + sym
    w = orc.normal_weights(N * K, seed) * 0.02
    if not sym:
        w = w + 0.01  # off-centre groups: zero-points away from 8
    p = orc.quantize(w, N, K, gs, sym)
    w_ref = orc.dequant_all(p)
    x = orc.normal_activations(M * K, seed + 1)
    dp = DevPacked(p)
    _check(c.gemm, dp.view, w_ref, x, M, N, K, seed)


@pytest.mark.parametrize("M,N,K", SHAPES)
def test_mxfp4_block(M, N, K):
    c = w4amd.capi()
    seed = M + N + K
    p = orc.quantize_mx(orc.outlier_weights(N, K, seed), N, K)
    w_ref = orc.dequant_all_mx(p)
    x = orc.normal_activations(M * K, seed + 1)
    dp = DevPackedMx(p)
    _check(c.gemm_mx, dp.view, w_ref, x, M, N, K, seed)


def test_block_shapes_add_in_one_order():
    """Rows at which the planner goes through blocks of 16 x 16 up to 64 x 96: K is split over the waves
    in the same way in all of them, so a row of the product has the same bytes in every call."""
    c = w4amd.capi()
    K, N = 4096, 2048
    p = orc.quantize(orc.normal_weights(N * K, 9) * 0.02, N, K, 128, True)
    x = orc.normal_activations(600 * K, 10)
    dp, x_d = DevPacked(p), to_dev(x)
    full = None
    for M in (600, 448, 320, 200, 128, 100, 64, 32, 17, 9):
        out = halves(M * N, 0x7E00)
        c.gemm(dp.view, ptr(x_d), ptr(out), M, 0, 0)
        got = bits(out).reshape(M, N)
        full = got if full is None else full
        assert np.array_equal(got, full[:M]), M


@pytest.mark.parametrize("M,N,K", [(60, 2064, 384), (33, 528, 2176), (16, 4096, 2400), (200, 4096, 4224)])
@pytest.mark.parametrize("kind", ["mx", 32, 64, 128])
def test_last_group_near_the_largest_half(M, N, K, kind):
    """K ends inside a unit and the row's last group is the only one with weights near 65504: codes of
    other groups would overflow with its scale, and nothing of the kind may reach the product."""
    c = w4amd.capi()
    rng = np.random.default_rng(M + K)
    gs = 32 if kind == "mx" else kind
    first = (K - 1) // gs * gs  # of the last group
    codes = rng.integers(0, 16, (N, K))
    if kind == "mx":
        codes[:, :first] |= 7                                    # +-6
        codes[:, first:] = rng.choice([0, 1, 2, 3, 4, 5, 9, 13], (N, K - first))  # up to +-3: 49152
    else:
        codes[:, first:] = rng.choice([7, 8, 9], (N, K - first))  # -1, 0, 1 times 60000
    words = (codes.reshape(N, K // 8, 8).astype(np.uint64) << (4 * np.arange(8, dtype=np.uint64))).sum(-1)
    x = orc.normal_activations(M * K, 3).view(np.float16).reshape(M, K).copy()
    x[:, first:] *= np.float16(2.0 ** -12)
    x = x.view(np.uint16).ravel()
    G = (K + gs - 1) // gs
    if kind == "mx":
        p = orc.quantize_mx(np.ones(N * K), N, K)
        s = np.full((N, G), 127 - 6, np.uint8)
        s[:, -1] = 127 + 14
        p.q[:], p.scales[:] = words.astype(np.uint32).ravel(), s.ravel()
        dp, fn, w_ref = DevPackedMx(p), c.gemm_mx, orc.dequant_all_mx(p)
    else:
        p = orc.quantize(np.ones(N * K), N, K, gs, True)
        s = np.full((N, G), 0.01, np.float16)
        s[:, -1] = 60000
        p.q[:], p.scales[:] = words.astype(np.uint32).ravel(), s.view(np.uint16).ravel()
        dp, fn, w_ref = DevPacked(p), c.gemm, orc.dequant_all(p)
    _check(fn, dp.view, w_ref, x, M, N, K, K)


@pytest.mark.parametrize("M,N,K,gs,sym", [(9, 2048, 4096, 128, True), (32, 4096, 4096, 128, False), (17, 8192, 8192, 256, True),
                                          (32, 8192, 8192, 128, False), (24, 528, 4352, 4352, True), (200, 4096, 4224, 128, True),
                                          (333, 4080, 4096, 128, False)])
def test_whole_chunk_groups_keep_their_scales_out_of_fp16(M, N, K, gs, sym):
    """Groups of whole 128-k chunks: (q - z) s is not rounded to FP16 before the sum, so an output is the
    product in FP64 rounded once, but where FP32 sums (some 1e-6 of the norm) end on the other side of a
    rounding boundary (ulp 5e-4 to 1e-3 of the value): one or two per cent of them.  Weights rounded first
    (1.7e-4 of the norm) move more than a quarter of the outputs."""
    rng = np.random.default_rng(M)
    w = orc.normal_weights(N * K, M + N) * 0.02 + (0.0 if sym else 0.01)
    p = orc.quantize(w, N, K, gs, sym)
    x = orc.normal_activations(M * K, 3)
    dp, x_d, out = DevPacked(p), to_dev(x), halves(M * N)
    w4amd.capi().gemm(dp.view, ptr(x_d), ptr(out), M, 0, 0)
    ns = np.unique(rng.choice(N, size=200))
    sh = 4 * np.arange(8, dtype=np.uint32)
    q = ((p.q.reshape(N, -1)[ns][:, :, None] >> sh) & 15).reshape(len(ns), -1)[:, :K].astype(np.float64)
    z = 8.0 if sym else ((p.zeros.reshape(N, -1)[ns][:, :, None] >> sh) & 15).reshape(len(ns), -1)[:, np.arange(K) // gs].astype(np.float64)
    s = p.scales.reshape(N, -1)[ns].view(np.float16).astype(np.float64)[:, np.arange(K) // gs]
    exact = x.view(np.float16).reshape(M, K).astype(np.float64) @ ((q - z) * s).T
    got = np.ascontiguousarray(bits(out).reshape(M, N)[:, ns])
    moved = np.mean(got != exact.astype(np.float16).view(np.uint16))
    assert moved <= 0.04, moved


# every block of every format: M ends inside a block and inside a row tile, N inside a block, K inside a unit
# (1152, 2176: after its first chunk; 2336, 2400: inside a chunk)
BLOCKS = [
    (11, 89, 256, 1152), (21, 227, 272, 2176), (22, 401, 272, 2336), (22, 276, 528, 2336), (24, 373, 528, 2336), (24, 377, 1040, 2336),
    (34, 409, 1040, 2400), (41, 75, 2720, 1152), (41, 345, 272, 2336), (42, 91, 4192, 1152), (42, 406, 528, 2336),
    (44, 412, 1568, 2336), (45, 391, 2160, 2336), (46, 403, 2608, 2336)]


@pytest.mark.parametrize("fmt,gs", [(0, 32), (0, 64), (0, 128), (1, 32), (1, 64), (1, 128), (2, 32)])
@pytest.mark.parametrize("block,M,N,K", BLOCKS)
def test_every_block(block, M, N, K, fmt, gs):
    c = w4amd.capi()
    got = c.gemm_plan_for(fmt, M, N, K, gs)
    if got != block:  # four of the blocks need other sizes with MXFP4, whose costs differ
        assert (fmt == 2 or block in (22, 24, 41, 42)) and got > 10, (got, block)
        return
    seed = M + N + K + gs + fmt
    x = orc.normal_activations(M * K, seed + 1)
    if fmt == 2:
        p = orc.quantize_mx(orc.outlier_weights(N, K, seed), N, K)
        dp = DevPackedMx(p)
        return _check(c.gemm_mx, dp.view, orc.dequant_all_mx(p), x, M, N, K, seed)
    p = orc.quantize(orc.normal_weights(N * K, seed) * 0.02 + 0.01 * fmt, N, K, gs, fmt == 0)
    dp = DevPacked(p)
    _check(c.gemm, dp.view, orc.dequant_all(p), x, M, N, K, seed)


def test_every_block_is_listed():
    """Each block of each format, with groups inside a chunk and with whole chunks, is one that the test above runs."""
    plan = w4amd.capi().gemm_plan_for
    for fmt, gs in [(0, 32), (0, 64), (0, 128), (1, 32), (1, 64), (1, 128), (2, 32)]:
        seen = {block for block, M, N, K in BLOCKS if plan(fmt, M, N, K, gs) == block}
        assert seen == {11, 21, 22, 24, 34, 41, 42, 44, 45, 46}, (fmt, gs, seen)


def test_plan_lines():
    """Where blocks measured slower than the kernel before them that kernel has the call, and the other way
    round: (format, M, N, K, gs) on both sides of the lines."""
    plan = w4amd.capi().gemm_plan_for
    other = [(0, 3, 128, 5120, 128), (0, 3, 4096, 6144, 64), (0, 7, 1024, 4224, 128), (0, 11, 128, 2304, 64),
             (0, 14, 1024, 4096, 128), (2, 3, 128, 4224, 32), (0, 4, 11008, 13824, 64), (0, 3, 11008, 6144, 32),
             (0, 17, 3952, 1920, 128), (0, 42, 2800, 1152, 64), (0, 72, 8192, 1152, 128), (2, 146, 6144, 2304, 32),
             (2, 2857, 288, 11904, 32), (2, 1256, 544, 4608, 32), (0, 984, 8192, 1088, 64), (0, 895, 8192, 5120, 96),
             (0, 28, 8736, 512, 128), (0, 12, 4096, 4096, 128), (0, 236, 28672, 1088, 128), (2, 503, 16384, 1088, 32)]
    assert [a for a in other if plan(*a) > 9] == []
    blocks = [(2, 50, 4096, 14336, 32), (1, 333, 4096, 4096, 64), (0, 16, 4096, 14336, 128), (0, 128, 4096, 4096, 128),
              (0, 64, 5120, 13824, 128), (0, 448, 3072, 9760, 128), (0, 7, 4096, 13824, 64), (2, 12, 8192, 8192, 32),
              (0, 12, 4096, 4096, 64), (0, 667, 13824, 5120, 96), (1, 1140, 5120, 13824, 96), (0, 89, 4096, 1152, 128), (1, 82, 6560, 1664, 32)]
    assert [a for a in blocks if plan(*a) < 10] == []
