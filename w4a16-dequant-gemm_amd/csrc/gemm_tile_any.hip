// The large-M W4A16 / MXFP4 GEMM of tile_dma.cuh for weights whose groups do not tile a 128-k stage: any
// group size and any K that are multiples of 8 (mma.cuh:63-230, the reference's kernel, takes them all).
#include <algorithm>

#include "tile_dma.cuh"

namespace w4k {
namespace {

// Whether a tile has two sets of waves, each on one half of K.
constexpr bool any_two_sets(int gsm, int shape) { return shape == 4 || (shape == 2 && gsm != 4); }

// shape: 0 = 128 x 256 (rows of X x rows of W), 2 = 64 x 128, 3 = 128 x 128, 4 = 32 x 128.  Hooked calls have the third
// only and split their sum over K where the unhooked call's tile does: both return the same bytes.
template <int FMT, int GSM, int KT>
hipError_t any_go(const WView& v, const w4_half* x, w4_half* c, w4_half* w_out, int M, hipStream_t s, int tn, int tm, int shape,
                  uint32_t mul) {
  if (w_out) {
    const int split_at = any_two_sets(GSM, shape) ? ((v.K + 127) / 128 + 1) / 2 : v.K;
    return launch<FMT, GSM, true, 128, 128, 1, KT>(v, x, c, w_out, M, s, (v.N + 127) / 128, (M + 127) / 128, split_at, mul);
  }
  if (shape == 4) return launch<FMT, GSM, false, 32, 128, 2, KT>(v, x, c, nullptr, M, s, tn, tm, 0, mul);
  if constexpr (GSM == 4) {
    static_assert(!any_two_sets(4, 2) && any_two_sets(3, 2), "one set for small groups");
    if (shape == 2) return launch<FMT, GSM, false, 64, 128, 1, KT>(v, x, c, nullptr, M, s, tn, tm, 0, mul);
  } else {
    if (shape == 2) return launch<FMT, GSM, false, 64, 128, 2, KT>(v, x, c, nullptr, M, s, tn, tm, 0, mul);
    if (shape == 0) return launch<FMT, GSM, false, 128, 256, 1, KT>(v, x, c, nullptr, M, s, tn, tm, 0, mul);
  }
  return launch<FMT, GSM, false, 128, 128, 1, KT>(v, x, c, nullptr, M, s, tn, tm, 0, mul);
}

// Time of a call in units of 10 ns: start + rounds of workgroups x (round + per_n x n) + store, n in stages of 128 k. Fitted to 6657
// shapes of 3 to 4000 rows, K = 256 to 14336, to within 4 to 10 % (r.m.s.); per_n: [symmetric W4, with zero-points,
// MXFP4], small: the same for groups of less than 32; store: what the outputs take, [N a multiple of 4 or not: halves one by one][the first
// round, or the part that is begun; a further one] (M = 3052, N = 2271, K = 256 25.1 us), fitted to 4600 shapes.
struct AnyShape {
  int shape, tm, tn, start, round, per_n[3], small_round, small_n[2], store[2][2];
};
constexpr AnyShape ANY_SHAPES[] = {{4, 32, 128, 130, 285, {57, 66, 43}, 290, {71, 88}, {{60, 0}, {245, 200}}},
                                   {2, 64, 128, 20, 430, {70, 74, 55}, 300, {98, 117}, {{140, 200}, {505, 500}}},
                                   {3, 128, 128, -70, 490, {105, 115, 90}, 510, {115, 133}, {{300, -60}, {960, 650}}},
                                   {0, 128, 256, -270, 850, {170, 186, 148}, 0, {0, 0}, {{560, -160}, {1860, 1090}}}};

// Whether the tile kernels for any group take the operands, their alignment apart.
bool any_applies(const WView& v, int M) {
  if (v.K < 128 || v.K % 8 || v.K >= 1 << 24) return false;
  if ((long long)v.N * v.K / 2 >= (1LL << 32) || (long long)M * v.K * 2 >= (1LL << 32)) return false;
  if ((long long)((v.N + 127) / 128) * ((M + 31) / 32) > 0x7FFFFFFFLL) return false;
  if (v.mx) return true;  // (a row has four blocks: one dword of scales is there)
  return (long long)v.N * v.G >= 2 && (long long)v.N * v.G < (1LL << 31) && any_group_fits(v);
}

// The fastest tile and its time; -1: none.
int any_shape(const WView& v, int M, int cus, int* time) {
  const bool rag = v.K % 32 != 0, small = !v.mx && v.gs < 32;
  const int stages = (v.K + 127) / 128, f = v.mx ? 2 : v.symmetric ? 0 : 1;
  int best = -1;
  long long least = 0;
  for (const AnyShape& s : ANY_SHAPES) {
    if (small && s.shape == 0) continue;  // (its parameters would not fit LDS)
    const long long tiles = (long long)((v.N + s.tn - 1) / s.tn) * ((M + s.tm - 1) / s.tm), rounds = (tiles + cus - 1) / cus;
    // (dword loads of codes: a tenth more)
    const long long per = (long long)(small ? s.small_n[f] : s.per_n[f]) * stages * (rag ? 11 : 10) / 10;
    const int* const store = s.store[v.N % 4 != 0];
    const long long out = tiles < cus ? tiles * store[0] / cus : store[0] + (tiles - cus) * store[1] / cus;
    const long long t = s.start + rounds * ((small ? s.small_round : s.round) + per) + out;
    if (best < 0 || t < least) best = s.shape, least = t;
  }
  *time = least > 1 << 30 ? 1 << 30 : (int)least;
  return best;
}

// Time of the kernel that has the call otherwise, in the same units: start + per_n x n + share x (share_0 + share_n x n).  n: steps of a
// wave (K-split kernel: chunks of 128 k; stream kernel: chunks, or pairs of them up to 32 rows, as many as its ring
// takes at a time), share: rounds of workgroups after the first (stream kernel: workgroups a compute unit has).  Rows of codes
// that are whole 16-byte pieces are loaded so and take 0.25 to 0.7 of the others' time.  Fitted to 14000 shapes of 5 to 4000
// rows, K = 64 to 14336, to within 6 to 13 % in whole pieces and 9 to 18 % otherwise (r.m.s.).
struct OtherShape {
  int start, per_n, share_0, share_n;
};
// [whole pieces][MXFP4, groups of whole slices of 32 k, other groups]
constexpr OtherShape OTHER_KSPLIT[2][3] = {{{210, 149, -304, 330}, {204, 158, -290, 312}, {171, 196, -348, 390}},
                                           {{298, 64, -106, 110}, {300, 73, -110, 114}, {223, 144, -164, 180}}};
// up to 32 rows: eight waves that share K by four (fewer than 128 workgroups of 64 rows of W) or by two
constexpr OtherShape OTHER_STREAM_BY4[2][3] = {{{180, 316, -24, 200}, {135, 379, 81, 133}, {202, 450, 5, 222}},
                                               {{224, 196, 86, 18}, {237, 207, 8, 62}, {191, 388, 103, 6}}};
constexpr OtherShape OTHER_STREAM_BY2[2][3] = {{{100, 375, 150, 20}, {146, 415, 25, 14}, {193, 518, -21, 19}},
                                               {{261, 134, 3, 23}, {257, 129, -36, 66}, {150, 380, 80, -20}}};
constexpr OtherShape OTHER_STREAM64[2][3] = {{{213, 76, -18, 239}, {251, 76, 0, 260}, {218, 115, -38, 306}},
                                             {{251, 44, 27, 150}, {273, 46, 29, 168}, {230, 96, 4, 221}}};
// The register-staged tiles of 256 x 128: start + (n + share x begun round) x k + further rounds x (round + round_n x k), k in
// steps of 64; 1, 2 or 4 steps in flight (fitted to 3200 shapes, to within 7 to 13 %).
constexpr int OTHER_TILE[3][5] = {{470, 124, 65, 510, 175}, {480, 101, 65, 600, 135}, {560, 84, 50, 650, 107}};

int other_time(const WView& v, int M, int cus) {
  const int chunks = (v.K + 127) / 128, cpw = (chunks + 7) / 8;
  const long long tiles = (v.N + 15) / 16;
  if (decode_general_applies(v, nullptr, nullptr, M)) {
    const int mt = M <= 16 ? 1 : M <= 32 ? 2 : 4, per = (v.gs < 32 ? 9 : 0) + (v.symmetric ? 64 : 74);
    return (int)(400 + (tiles + cus - 1) / cus * (cpw * (per + 19 * mt) - 30));
  }
  const bool pieces = v.K % 32 == 0, halves = v.N % 4 != 0;  // (halves: outputs are stored one by one)
  long long t;
  if (M >= 96 && v.K % 64 == 0) {
    const int k = v.K / 64, *const c = OTHER_TILE[(!v.mx && v.gs % 16) || k % 2 ? 0 : k % 4 ? 1 : 2];
    const long long wgs = (long long)((v.N + 127) / 128) * ((M + 255) / 256), more = (wgs + cus - 1) / cus - 1;
    const long long part = wgs < cus ? wgs * 64 / cus : 64;  // of the first round, in 64ths
    t = c[0] + (c[1] * 64 + c[2] * part) * k / 64 + more * (c[3] + c[4] * k);
    if (halves) t += 430 + 500 * part / 64 + 700 * more;
  } else {
    const int form = v.mx ? 0 : v.gs % 32 == 0 ? 1 : 2;
    const OtherShape* c = &OTHER_STREAM64[pieces][form];
    int n = cpw;
    long long share, whole = 64, more_rows = 0;  // share, whole: in 64ths
    if (M <= 8 || (M <= 16 && v.N < 8192)) {
      c = &OTHER_KSPLIT[pieces][form];
      share = 64 * ((tiles + cus - 1) / cus - 1);
      // (a second half of 16 rows: N = 2874, K = 4096, gs = 32 with zero-points, M = 15 8.4 us, 5.9 without the term)
      if (M > 8 && n > 8) more_rows = 100 * (n - 8);
      if (M > 8 && n > 2 && pieces) more_rows += 30 * std::min(n, 8);
    } else {
      long long wgs = (long long)((v.N + 63) / 64) * ((M + 63) / 64);
      if (M <= 32) {
        const bool by4 = wgs < 128;
        c = by4 ? &OTHER_STREAM_BY4[pieces][form] : &OTHER_STREAM_BY2[pieces][form];
        n = ((chunks + 1) / 2 + (by4 ? 3 : 1)) / (by4 ? 4 : 2);
        if (n >= 2) n = (n + 1) / 2 * 2;
        if (by4) wgs = (v.N + 31) / 32;
      } else {
        n = (chunks + 1) / 2;
        if (n >= 4) n = (n + 3) / 4 * 4;
      }
      share = 2 * wgs > cus ? wgs * 64 / cus : 32;
      // (up to 32 rows the shapes end at N = 16384, a workgroup a compute unit: on from there all but the start grows)
      if (M <= 32 && share > 64) whole = share;
    }
    t = c->start + more_rows + whole * c->per_n * n / 64 + share * (c->share_0 + c->share_n * n + (halves && M > 32 ? 110 : 0)) / 64;
    // (a word's zero-point in small groups: 1.2 to 1.4 of the time in the stream kernels, N = 9712, K = 1024, gs = 8, M = 53 20.0 us,
    // tiles 11.1)
    if (pieces && !v.mx && !v.symmetric && v.gs < 32 && c != &OTHER_KSPLIT[pieces][form]) t = t * 5 / 4;
  }
  return t > 1 << 30 ? 1 << 30 : (int)t;
}

// What the general decode kernel takes on top of that: next to the activations of 33 to 64 rows LDS has room for the
// parameters of one or two tiles of small groups, so that there are further rounds of workgroups, each of which fetches the
// activations again: 3.5 us with one tile, 0.9 with two (one tile: 1.17 to 1.44 of the time above, 0.96 to 1.04 of the sum).
int general_rounds(const WView& v, int M, int cus) {
  if (v.mx || v.gs >= 32 || M <= 32) return 0;
  const int held = decode_general_tiles(v, M);
  if (!held) return 0;
  const long long tiles = (v.N + 15) / 16, rounds = ((tiles + held - 1) / held + cus - 1) / cus;
  return (int)((rounds - 1) * (held == 1 ? 350 : 90));
}

// By how much blocks and tiles have to be ahead of the kernel before: a twelfth of that kernel's time, but no more than 0.67 us,
// about the error of the times.  Of 6009 random shapes with N, K >= 1024, all three kernels timed, 147 take more than 1.1 of the
// best one's time with an eighth, 136 with a twelfth and 144 with a sixteenth; 69, 74 and 89 more than 1.05 of the kernel before's.
int any_lead(int other) { return std::min(other, 800) / 12; }

}  // namespace

bool any_group_fits(const WView& v) { return v.mx || (long long)(v.K / 8) * (v.gs / 8) < (1LL << 31); }

AnyPlan any_plan(const WView& v, int M) {
  const AnyPlan none{0, -1};
  if (M < 5 || v.K % 8) return none;
  const int cus = device_cus();
  if (cus < 8) return none;
  // Shorter rows are no more than a launch for the kernels that have them.  Up to 16 rows on few tiles: N < 2048, K = 1281 to
  // 3072 0.83 to 1.0 times as fast, up to 4096 1.05 to 1.13; N = 2048 to 4096, K up to 2048 0.9 to 1.03.
  const int tiles = (v.N + 15) / 16;
  if (v.K < (M >= 17 ? 256 : 2 * tiles < cus ? 3073 : tiles <= cus ? 2049 : 1152)) return none;
  const bool dma = v.K % 128 == 0 && (v.mx || v.gs == 32 || v.gs == 64 || v.gs % 128 == 0);
  const bool whole = v.N % 16 == 0 && v.K % 32 == 0 && (v.mx || v.gs % 32 == 0);
  // shapes of the kernels for whole tiles, chunks and groups
  if (whole && (M < 17 || (v.K % 128 == 0 && M <= 64))) return none;
  // the direct-to-LDS tiles take any N (but no fewer than eight tiles, and no scales that end inside a dword)
  if (dma && M >= 65 && (long long)((v.N + 255) / 256) * ((M + 127) / 128) >= 8 &&
      (v.mx || v.gs < 128 || (long long)v.N * v.G % 2 == 0)) return none;
  int tile = -1, tile_time = 1 << 30, block_shape = -1, block_t = 1 << 30;
  if (any_applies(v, M)) tile = any_shape(v, M, cus, &tile_time);
  if (whole) {
    // blocks as block_plan() has them; tiles where these take less than 0.85 of the time (up to there 3 of 380 calls lost: M = 157,
    // N = 9904, K = 12768, gs = 32 with zero-points 92 us in blocks and 105 on tiles; as many again gained 20 % between 0.75 and 0.85)
    block_shape = block_plan_time(v, M, &block_t);
    // (W4 groups of whole chunks: blocks scale a chunk's FP32 sums, tiles round every weight; 2.1e-4 and 2.7e-4 from the
    // product in FP64)
    if (block_shape >= 0 && !v.mx && v.gs % 128 == 0) return AnyPlan{1, block_shape};
    if (block_shape < 0) {
      if (decode_resident_applies(v, nullptr, nullptr, M)) return AnyPlan{3, -1};
      const int other = other_time(v, M, cus);
      return tile_time < other - any_lead(other) ? AnyPlan{2, tile} : AnyPlan{3, -1};
    }
    return 20LL * tile_time < 17LL * block_t ? AnyPlan{2, tile} : AnyPlan{1, block_shape};
  }
  block_shape = block_any_time(v, M, cus, &block_t);
  const bool general = !v.mx && decode_general_applies(v, nullptr, nullptr, M);
  const int other = other_time(v, M, cus), rounds = (int)std::min((long long)other + general_rounds(v, M, cus), 1LL << 30);
  // (tiles are asked to beat that kernel's time without its further rounds: 33 to 64 rows of small groups take them 0.95 to
  // 1.4 times that kernel's time, and blocks 0.65 to 0.9; N = 11008, gs = 8, M = 64: K = 4096 29.2 -> 24.5 us)
  // Up to five rounds of its tiles they have to be ahead by a quarter: M = 41, N = 11504, K = 2176, gs = 8 13.1 us there and 18.3
  // on tiles, M = 54, N = 13936, K = 2752 18.1 and 21.6; past them M = 40, N = 28672, K = 4096 55 and 42.
  const bool close = general && v.gs < 32 && M > 32 && tiles <= 5 * cus;
  // Otherwise blocks and tiles have to be ahead by any_lead().
  const bool tiles_ahead = close ? 4LL * tile_time < 3LL * other : tile_time < other - any_lead(other);
  const bool blocks_ahead = block_t < rounds - any_lead(rounds);
  if (!tiles_ahead && !blocks_ahead) return none;
  // (with tiles up to 0.95, 1 and 1.05 of the blocks' time 259, 228 and 229 of 8000 calls take more than 1.1 of the best time)
  return tiles_ahead && (!blocks_ahead || tile_time < block_t) ? AnyPlan{2, tile} : AnyPlan{1, block_shape};
}

bool try_tile_any(const WView& v, const w4_half* x, w4_half* c, int M, hipStream_t s, w4_half* w_out, int shape,
                  hipError_t* err) {
  const bool rag = v.K % 32 != 0;
  if (((uintptr_t)x & 15) || ((uintptr_t)v.q & (rag ? 3 : 15)) || ((uintptr_t)v.scales & 3)) return false;
  if ((!v.mx && !v.symmetric && ((uintptr_t)v.zeros & 3)) || ((uintptr_t)w_out & 15)) return false;
  const int TN = shape == 0 ? 256 : 128, TM = shape == 2 ? 64 : shape == 4 ? 32 : 128;
  const int tn = (v.N + TN - 1) / TN, tm = (M + TM - 1) / TM;
  const uint32_t mul = v.mx ? 0u : (uint32_t)(((1ULL << 31) + v.gs / 8 - 1) / (v.gs / 8));
#define W4_GO(F, G) (rag ? any_go<F, G, 2>(v, x, c, w_out, M, s, tn, tm, shape, mul) : any_go<F, G, 1>(v, x, c, w_out, M, s, tn, tm, shape, mul))
  if (v.mx) *err = W4_GO(2, 3);
  else if (v.symmetric) *err = v.gs >= 32 ? W4_GO(0, 3) : W4_GO(0, 4);
  else *err = v.gs >= 32 ? W4_GO(1, 3) : W4_GO(1, 4);
#undef W4_GO
  return true;
}

}  // namespace w4k
