// The W4A16 / MXFP4 GEMM for large M whose operands reach LDS directly (tile_dma.cuh): tile shapes and
// the rule that picks one, for weights whose groups tile a 128-k stage.
#include "tile_dma.cuh"

namespace w4k {
namespace {

// shape: 0 = 128 x 256 (rows of X x rows of W), 1 = 64 x 256, 2 = 64 x 128, 3 = 128 x 128,
// 4 = 32 x 128 (the hooked kernels exist for the first only)
// sets: 2 = the small tiles with two sets of waves (the hooked kernel then splits its sum at
// split_at, the first stage of the second set)
template <int FMT, int GSM>
hipError_t launch_hook(const WView& v, const w4_half* x, w4_half* c, w4_half* w_out, int M,
                       hipStream_t s, int tn, int tm, int shape, int sets, int split_at) {
  if (w_out) return launch<FMT, GSM, true, 128, 256>(v, x, c, w_out, M, s, tn, tm, split_at);
  const int none = v.K;  // more than any stage index
  if (shape == 4 && sets == 2) return launch<FMT, GSM, false, 32, 128, 2>(v, x, c, nullptr, M, s, tn, tm, none);
  if (shape == 2 && sets == 2) return launch<FMT, GSM, false, 64, 128, 2>(v, x, c, nullptr, M, s, tn, tm, none);
  if (shape == 4) return launch<FMT, GSM, false, 32, 128>(v, x, c, nullptr, M, s, tn, tm, none);
  if (shape == 3) return launch<FMT, GSM, false, 128, 128>(v, x, c, nullptr, M, s, tn, tm, none);
  if (shape == 2) return launch<FMT, GSM, false, 64, 128>(v, x, c, nullptr, M, s, tn, tm, none);
  if (shape == 1) return launch<FMT, GSM, false, 64, 256>(v, x, c, nullptr, M, s, tn, tm, none);
  return launch<FMT, GSM, false, 128, 256>(v, x, c, nullptr, M, s, tn, tm, none);
}

template <int FMT>
hipError_t launch_gsm(int gsm, const WView& v, const w4_half* x, w4_half* c, w4_half* w_out,
                      int M, hipStream_t s, int tn, int tm, int shape, int sets, int split_at) {
  if (gsm == 0) return launch_hook<FMT, 0>(v, x, c, w_out, M, s, tn, tm, shape, sets, split_at);
  if (gsm == 1) return launch_hook<FMT, 1>(v, x, c, w_out, M, s, tn, tm, shape, sets, split_at);
  return launch_hook<FMT, 2>(v, x, c, w_out, M, s, tn, tm, shape, sets, split_at);
}

}  // namespace

// Takes MXFP4 weights and W4 weights whose groups tile a 128-k stage (gs 32, 64 or a
// multiple of 128), M >= 65, K a multiple of 128, operands under 4 GiB (32-bit offsets),
// 16-byte aligned rows, scales that can be fetched as aligned dwords, and at least
// eight tiles (measured at N = K = 4096: M = 128, 16 tiles, 44 us against 56 us for
// the register-staged kernel).  Returns false, launching nothing, otherwise.
bool try_tile_dma(const WView& v, const w4_half* x, w4_half* c, int M, hipStream_t s,
                  w4_half* w_out, hipError_t* err) {
  if (v.K % 128 || v.K < 128) return false;
  int gsm = 2;
  if (!v.mx) {
    if (v.gs % 128 == 0) gsm = 0;
    else if (v.gs == 64) gsm = 1;
    else if (v.gs != 32) return false;
  }
  // The smallest of the tile shapes whose grid still fits the chip's 256 compute
  // units in one round: a smaller tile shortens a workgroup's walk over K -- N = K =
  // 4096, M = 512: 45.6 us with 128 x 256 tiles, 38.1 with 64 x 256, 27.0 with 64 x 128;
  // M = 256: 23.7 with 64 x 128 (128 workgroups), 21.8 with 32 x 128 (256).  On such grids a
  // workgroup's K / 128 stages are a chain of 0.6 - 0.7 us each whatever the tile holds.
  // (Hooked
  // and unhooked calls add in the same order whatever the shape: a wave's sums do
  // not depend on how many rows its workgroup holds.)
  const long long n256 = (v.N + 255) / 256, n128 = (v.N + 127) / 128;
  const long long m128 = (M + 127) / 128, m64 = (M + 63) / 64, m32 = (M + 31) / 32;
  // the shape an unhooked call takes; the hooked kernel has 128 x 256 tiles only, but follows
  // the unhooked call's split of the sum over K (below)
  // Groups of 32 with zero-points have three dwords of parameters a row and stage, which 128 rows of W a workgroup cannot
  // fetch here: the two smallest tiles are those of the kernels for any group (N = 1639, K = 6784, M = 136
  // 61.3 -> 40.2 us; N = K = 4096, M = 512 37.7 -> 32.3; N = K = 5120, M = 300 46.2 -> 35.7).
  const bool planes3 = gsm == 2 && !v.mx && !v.symmetric;
  int shape = 0;
  {
    if (n128 * m32 <= 256) shape = 4;
    else if (n128 * m64 <= 256) shape = 2;
    else if (!planes3 && n128 * m128 <= 256) shape = 3;
    else if (n256 * m64 <= 256) shape = 1;
  }
  // The two smallest tiles run with two sets of waves, each on one half of K (their stages
  // are a serial chain; see the kernel): the sum over K is then (first half) + (second half).
  const int stages = v.K / 128;
  const bool any = planes3 && (shape == 2 || shape == 4);
  const int any_tile = shape;
  const int sets = (shape == 2 || shape == 4) && (stages >= 8 || any) ? 2 : 1;
  const int split_at = sets == 2 ? (stages + 1) / 2 : v.K;
  if (w_out) shape = 0;
  const long long tiles_n = (shape == 2 || shape == 3 || shape == 4) ? n128 : n256;
  const long long tiles_m = (shape == 0 || shape == 3) ? m128 : shape == 4 ? m32 : m64;
  if (M < 65 || n256 * m128 < 8 || tiles_n * tiles_m > 0x7FFFFFFFLL) return false;
  if ((long long)v.N * v.K / 2 >= (1LL << 32) || (long long)M * v.K * 2 >= (1LL << 32)) return false;
  // one FP16 scale per stage: the dword around it must lie inside the array
  if (gsm == 0 && (((long long)v.N * v.G) & 1)) return false;
  if ((((uintptr_t)v.q | (uintptr_t)x) & 15) || ((uintptr_t)v.scales & 3)) return false;
  if (!v.mx && !v.symmetric && (v.zeros == nullptr || ((uintptr_t)v.zeros & 3))) return false;
  if (w_out && ((uintptr_t)w_out & 15)) return false;
  // grids of more than one round: 256 x 256 tiles where they halve the rounds
  if (!w_out && try_tile256(v, x, c, M, s, 256, err)) return true;
  if (any && !w_out) return try_tile_any(v, x, c, M, s, nullptr, any_tile, err);
  const int tn = (int)tiles_n, tm = (int)tiles_m;
  if (v.mx) *err = launch_hook<2, 2>(v, x, c, w_out, M, s, tn, tm, shape, sets, split_at);
  else if (v.symmetric) *err = launch_gsm<0>(gsm, v, x, c, w_out, M, s, tn, tm, shape, sets, split_at);
  else *err = launch_gsm<1>(gsm, v, x, c, w_out, M, s, tn, tm, shape, sets, split_at);
  return true;
}

}  // namespace w4k
