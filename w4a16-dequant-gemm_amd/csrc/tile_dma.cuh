// Large-M W4A16 GEMM whose operands reach LDS without passing through registers:
// c[M,N] = X[M,K] * dequant(W)[N,K]^T for W4 weights with FP16 group scales and
// optional 4-bit zero-points (mma.cuh:63-230 is the reference's tensor-core kernel:
// it expands each chunk of W to FP16 in shared memory once per block).
//
// Here the packed words themselves are what sits in LDS -- a quarter of the bytes
// of the expanded tile -- and every wave expands the words of its own MFMA
// operands in registers, straight into the operand layout:
//   * global_load_lds_dwordx4 moves both operand tiles global -> LDS (no staging
//     registers, no ds_write); a stage is 128 k: 64 bytes of a W row, 256 bytes of
//     an X row; three stages of 50 KB; one barrier per stage.
//   * v_mfma_f32_32x32x16_f16: lane l brings row l%32 and eight consecutive k.
//     Which eight is free as long as both operands agree, so of a 64-k half lane
//     half h = l/32 takes k 32h + 8j .. + 7 in MFMA j: its four W words are one
//     16-byte LDS read, its X operand is 16-byte piece 4h + j of the row's half.
//   * a word becomes four packed-half registers in natural k order with
//     v_perm_b32 (byte i to bytes 0 and 2), one mask-and-or that plants the low
//     nibble in the significand of 1024.0 and the high nibble in that of 64.0
//     (whose unit in the last place is 1/16), one packed add of -(1024 + z),
//     -(64 + z) and one packed multiply by the scale: q - z is exact and the
//     product is rounded once, so the operand is bit for bit the FP16 weight the
//     one dequant step returns (pack.hpp:58-60).
// The accumulation is FP32 in the instruction; the output is rounded to FP16 once.
#pragma once

#include <atomic>

#include "dq.cuh"
#include "kernels.h"

namespace w4k {
namespace {

typedef float f16v __attribute__((ext_vector_type(16)));
typedef __attribute__((address_space(3))) void* lds_ptr;

// rows of W (TN: 256 or 128) and of X (TM: 128, 64 or 32) per workgroup are template parameters
constexpr int TD_WAVES = 4, TD_THREADS = 64 * TD_WAVES;  // a wave: 64 rows of W x all 128 of X
constexpr int TD_STAGES = 3;
// a stage: TN rows of W (64 bytes each), TM rows of X (256 bytes each), two scale dwords and a
// zero-point word per W row
constexpr int td_tile(int tm, int tn) { return tn * 64 + tm * 256; }
constexpr int td_stage(int tm, int tn, int planes = 3) { return td_tile(tm, tn) + planes * tn * 4; }
constexpr int td_lds_bytes(int tm, int tn, int planes = 3) { return TD_STAGES * td_stage(tm, tn, planes); }
// (KT > 0: a slice's run is read as whole dwords, of which the last may be one more than a stage has: a dword a row further)
constexpr int td_any_slack(int tn, int kt) { return kt ? tn * 4 : 0; }
// Parameter dwords per W row and stage of the kernels for any group (KT > 0): scales, then zero-points.
// 128 k that start at a multiple of 8 touch five groups of 32 or more k (gsm 3), sixteen of 8 (gsm 4) or five
// MXFP4 blocks, whose run starts at any half (MXFP4: byte) of the first dword.
constexpr int td_any_scales(int fmt, int gsm) { return fmt == 2 ? 2 : gsm == 3 ? 3 : 9; }
constexpr int td_any_zeros(int fmt, int gsm) { return fmt != 1 ? 0 : gsm == 3 ? 2 : 3; }
constexpr int td_planes(int fmt, int gsm, int kt) {
  return kt == 0 ? 3 : td_any_scales(fmt, gsm) + td_any_zeros(fmt, gsm);
}

extern __shared__ __attribute__((aligned(16))) uint8_t td_lds[];

// Position of 16-byte piece p of row R.  A load instruction writes lane l's 16
// bytes at 16 l, so the rows of one instruction are contiguous (16 rows of W, 4 of
// X) and the piece a lane fetches is chosen so that the rows one ds_read_b128
// touches (8 or 16 consecutive ones, same p) fall on distinct 16-byte bank groups.
__device__ __forceinline__ int w_key(int R) { return ((R >> 1) ^ (R >> 3)) & 3; }
__device__ __forceinline__ int w_at(int R, int p) {
  return (R >> 4) * 1024 + ((R & 15) * 4 + (p ^ w_key(R))) * 16;
}
__device__ __forceinline__ int x_at(int R, int p) {
  return (R >> 2) * 1024 + ((R & 3) * 16 + (p ^ (R & 15))) * 16;
}

// One wave per SIMD, so the three pipes have to overlap inside a wave: a stage is
// eight steps of 16 k (8 MFMAs each); during the MFMAs of step u the wave reads the
// X operands of step u + 1 from LDS and expands its W words, in program order
// between the MFMAs.
//
// HOOK: the workgroups of the first m tile also write the expanded weights to
// w_out (mma.cuh:147-159: the reference's dequant hook), from the operand
// registers the MFMAs consume.
//
// FMT: 0 W4 symmetric, 1 W4 with zero-points, 2 MXFP4.  GSM says how the groups
// lie in a 128-k stage: 0 one group (gs a multiple of 128), 1 two (gs = 64), 2 four
// (gs = 32, and the 32-blocks of MXFP4).  A lane's share of a 64-k half is 32
// consecutive k, so even then it has one scale per half.  G: scales per row.
// TM: rows of X per workgroup, 128, 64 or 32 (a wave: 64 rows of W x all TM of X).  The
// smaller tile halves a workgroup's walk over K when the grid of the larger one
// would leave most of the chip idle.
// TN: rows of W per workgroup, 256 or 128 (a wave: TN / 4 of them = NI tiles of 32).
// KG: sets of four waves per workgroup.  With two, each set walks one half of the K / 128
// stages through stage buffers of its own (two waves per SIMD, whose instruction streams
// interleave) and the second set's sums are added to the first set's at the end, through
// LDS: on the thin grids of the small tiles a workgroup's stages are a chain of 0.6 us
// each whatever they hold, and this halves the chain.  split_at: the hooked kernel, which
// always has one set, starts a second accumulator at that stage and adds the two at the
// end, so that it returns the bytes of the two-set kernel (no split: a stage past the last).
//
// KT: 0 = K a multiple of 128 and groups as GSM says.  Otherwise any group size and any K that are
// multiples of 8 (gsm 3: W4 groups of 32 or more k, or MXFP4; 4: smaller ones):
//   * the scales and zero-points that a stage touches come as a run of dwords per row (td_any_scales), from
//     which every word picks its own two by the group it lies in (group_mul: the divisor's reciprocal);
//   * the last stage is the row's last 128 k, whatever the stage before it ended at.  What both hold is
//     multiplied by the stage before: in the last stage its activations are cleared in LDS and its scale reads as 0;
//   * KT = 2: rows of words are 4-byte aligned only (K no multiple of 32) and come dword by dword.
template <int FMT, int GSM, bool HOOK, int TM, int TN, int KG, int KT>
__global__ __launch_bounds__(TD_THREADS * KG) void w4_tile_dma_kernel(
    const uint32_t* __restrict__ wq, const void* __restrict__ scales,
    const uint32_t* __restrict__ zeros, const w4_half* __restrict__ x, w4_half* __restrict__ c,
    w4_half* __restrict__ w_out, int N, int K, int G, int gs, int M, int tiles_n, int tiles_m,
    int split_at, uint32_t group_mul) {
  constexpr bool ASYM = FMT == 1, MX = FMT == 2;
  constexpr bool ANY = KT > 0;
  static_assert(!ANY || GSM >= 3, "the kernels for any group take parameters as runs");
  constexpr int NSC = (!MX && GSM == 2) ? 2 : 1;           // scale dwords per row and stage
  // ANY: a load instruction takes one dword of 64 rows.  The twelve of a row of small groups would hold up the thinnest
  // tile, whose stage is short: there neighbouring lanes take neighbouring dwords of a row (RUNS: N = 11008, K =
  // 4104, gs = 8, M = 32 39.8 -> 35.2 us; larger tiles lose by it, 128 x 256, gs = 48 433 -> 454).  The waves share
  // the loads out; a count that is no multiple of the waves repeats the last one.
  constexpr int PS = td_any_scales(FMT, GSM), PZ = td_any_zeros(FMT, GSM);
  constexpr bool RUNS = GSM == 4 && TM == 32;
  constexpr int SROW = RUNS ? PS * 4 : 4, SDW = RUNS ? 4 : TN * 4;  // bytes between rows, and between the dwords of one
  constexpr int ZROW = RUNS ? PZ * 4 : 4, ZDW = RUNS ? 4 : TN * 4;
  static_assert(!ANY || (SDW <= td_any_slack(TN, KT) && ZDW <= td_any_slack(TN, KT)), "what a slice reads ends inside LDS");
  constexpr int PSN = TN * PS / 64, PZN = TN * PZ / 64, PSI = (PSN + 3) / 4, PZI = (PZN + 3) / 4;
  constexpr int TD_TM = TM, MJ = TM / 32;                  // 32-row tiles of X per wave
  constexpr int TD_TN = TN, NI = TN / 128;                 // 32-row tiles of W per wave
  constexpr int TD_W_BYTES = TN * 64;
  constexpr int TD_WI = TD_W_BYTES / 1024 / TD_WAVES;      // 1 KB load instructions of W per wave
  constexpr int TD_TILE = td_tile(TM, TN), TD_STAGE = td_stage(TM, TN, td_planes(FMT, GSM, KT));
  constexpr int TD_XI = TM * 256 / 1024 / TD_WAVES;        // 1 KB load instructions of X per wave
  constexpr int WLOADS = KT == 2 ? 4 * TD_WI : TD_WI;      // load instructions of W per wave
  constexpr int LOADS = WLOADS + TD_XI + (ANY ? PSI + PZI : NSC + (ASYM ? 1 : 0));  // load instructions per wave and stage
  constexpr int PPS = ANY ? (LOADS + 7) / 8 : 2;           // ... issued per step
  static_assert(LOADS <= 8 * PPS && LOADS + PPS < 64, "a stage's requests fit its steps and the counter");
  constexpr bool PHASED = NI * MJ >= 4;  // a step has the four MFMAs that the phases of an expansion go under
  const int t = threadIdx.x, lane = t & 63;
  const int wave_all = __builtin_amdgcn_readfirstlane(t >> 6);  // in an SGPR: LDS addresses go to M0
  const int wave = KG == 2 ? (wave_all & 3) : wave_all;        // within its set of four
  const int grp = KG == 2 ? (wave_all >> 2) : 0;               // the set
  const int r = lane & 31, h = lane >> 5;
  // Consecutive workgroup ids land on different XCDs (each with its own L2): give
  // each XCD a contiguous run of the tile order, m fastest, so that its
  // workgroups share a few W tiles and walk X.
  int L = blockIdx.x;
  const int total = tiles_n * tiles_m;
  if (total % 8 == 0) L = (L & 7) * (total >> 3) + (L >> 3);
  const int n0 = (L / tiles_m) * TD_TN, m0 = (L % tiles_m) * TD_TM;
  const int wg = words(G);

  // What this lane fetches (byte offsets; 32 bits: the launcher bounds the operands).
  // Rows past N or M are clamped to the last one; their results are never stored.
  uint32_t wo[WLOADS], xo[TD_XI];
#pragma unroll
  for (int i = 0; i < WLOADS; ++i) {
    if constexpr (KT == 2) {  // four rows, a dword a lane, to the places that the 16-byte loads give them
      const int R = (wave + TD_WAVES * i) * 4 + (lane >> 4), n = n0 + R;
      wo[i] = (uint32_t)(n < N ? n : N - 1) * (uint32_t)(K >> 1) + ((((lane >> 2) & 3) ^ w_key(R)) * 16) + (lane & 3) * 4;
    } else {
      const int R = (wave + TD_WAVES * i) * 16 + (lane >> 2), n = n0 + R;
      wo[i] = (uint32_t)(n < N ? n : N - 1) * (uint32_t)(K >> 1) + (((lane & 3) ^ w_key(R)) * 16);
    }
  }
#pragma unroll
  for (int i = 0; i < TD_XI; ++i) {
    const int R = (wave + TD_WAVES * i) * 4 + (lane >> 4), m = m0 + R;
    xo[i] = (uint32_t)(m < M ? m : M - 1) * (uint32_t)(K * 2) + (((lane & 15) ^ (R & 15)) * 16);
  }
  // per stage: the dword that holds the group scale of W row 64 wave + lane, and
  // (ASYM) that row's zero-point word
  // (TN = 128: waves 2 and 3 repeat the fetches of waves 0 and 1, which keeps the count of
  // load instructions the same for every wave)
  const int srow = (NI == 2 ? wave : (wave & 1)) * 64 + lane;
  const uint32_t sn = (uint32_t)(n0 + srow < N ? n0 + srow : N - 1);
  const uint32_t sc_base = sn * (uint32_t)G, zw_base = sn * (uint32_t)wg;
  [[maybe_unused]] uint32_t sb[PSI], zb[PZI > 0 ? PZI : 1];  // ANY: of this lane's dwords, in scales and words
  if constexpr (ANY) {
#pragma unroll
    for (int i = 0; i < PSI; ++i) {
      const int D = min(wave + TD_WAVES * i, PSN - 1) * 64 + lane, n = n0 + (RUNS ? D / PS : D % TN);
      sb[i] = (uint32_t)(n < N ? n : N - 1) * (uint32_t)G + (uint32_t)(RUNS ? D % PS : D / TN) * (MX ? 4u : 2u);
    }
    if constexpr (ASYM) {
#pragma unroll
      for (int i = 0; i < PZI; ++i) {
        const int D = min(wave + TD_WAVES * i, PZN - 1) * 64 + lane, n = n0 + (RUNS ? D / PZ : D % TN);
        zb[i] = (uint32_t)(n < N ? n : N - 1) * (uint32_t)wg + (uint32_t)(RUNS ? D % PZ : D / TN);
      }
    }
  }
  const char* wqb = (const char*)wq;
  const char* xb = (const char*)x;

  const int stages = ANY ? (K + 127) >> 7 : K >> 7;
  // ANY: first k of stage d (of the last one: K - 128), its group, and the words that the stage before it has
  [[maybe_unused]] auto first_k = [&](int d) { return (uint32_t)min(d * 128, K - 128); };
  [[maybe_unused]] auto group_of_word = [&](uint32_t w) { return MX ? w >> 2 : __umulhi(2u * w, group_mul); };
  [[maybe_unused]] const uint32_t overlap = ANY ? (uint32_t)(stages * 128 - K) >> 3 : 0u;
  [[maybe_unused]] const uint32_t sc_last = max(((uint32_t)N * (uint32_t)G) >> (MX ? 2 : 1), 1u) - 1u,
                                  zw_last = (uint32_t)N * (uint32_t)wg - 1u;
  // this set's stages: d_first .. d_first + per_set - 1, those below `stages` (both sets run
  // per_set iterations so that they meet at every barrier; a stage past the end is fetched
  // from the last one and not multiplied)
  const int per_set = (stages + KG - 1) / KG;
  const int d_first = grp * per_set;
  const int d_end = min(d_first + per_set, stages) > d_first ? min(d_first + per_set, stages) : d_first + 1;
  // The loads are asm so that the compiler neither tracks them (it would wait for
  // all of them before any LDS read) nor moves LDS reads across them; the vmcnt
  // waits below are by hand.  M0 carries the wave-uniform LDS address.
  auto dma16 = [](const void* gbase, uint32_t goff, uint32_t lds_addr, int lds_off) __attribute__((always_inline)) {
    asm volatile("s_add_u32 m0, %2, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
                 :
                 : "v"(goff), "s"(gbase), "s"(lds_addr), "i"(lds_off)
                 : "memory", "m0", "scc");
  };
  auto dma4 = [](const void* gbase, uint32_t goff, uint32_t lds_addr) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dword %0, %1"
                 :
                 : "v"(goff), "s"(gbase), "s"(lds_addr)
                 : "memory", "m0");
  };
  const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_ptr)td_lds;
  // Load instruction `part` (0 .. LOADS - 1) of stage d: a wave issues them two at
  // a time between the MFMAs of successive steps -- thirteen in a row would hold up
  // its one instruction stream for as long as four steps take.
  auto request_part = [&](int d, uint32_t buf, int part) {  // buf: byte offset of the stage's buffer
    const uint32_t dd = (uint32_t)(d < d_end ? d : d_end - 1);  // past the set's end: valid, never used
    const uint32_t st = lds0 + buf;
    const uint32_t k0 = ANY ? first_k((int)dd) : dd * 128u;
    if (part < WLOADS) {  // the stage's offset goes into the scalar base: no vector arithmetic
      if constexpr (KT == 2) dma4(wqb + (k0 >> 1), wo[part], st + (wave + TD_WAVES * part) * 256);
      else dma16(wqb + (k0 >> 1), wo[part], st + wave * 1024, TD_WAVES * part * 1024);
    } else if (part < WLOADS + TD_XI) {
      const int i = part - WLOADS;
      dma16(xb + k0 * 2u, xo[i], st + wave * 1024, TD_W_BYTES + TD_WAVES * i * 1024);
    } else if constexpr (ANY) {  // the runs of dwords that begin with the stage's first group
      const int k = part - WLOADS - TD_XI;
      const uint32_t g = group_of_word(k0 >> 3);
      if (k < PSI) {
        const uint32_t at = __builtin_amdgcn_readfirstlane(min(wave + TD_WAVES * k, PSN - 1) * 256);
        dma4(scales, min((sb[k < PSI ? k : 0] + g) >> (MX ? 2 : 1), sc_last) * 4u, st + TD_TILE + at);
      } else if constexpr (ASYM) {
        const uint32_t at = __builtin_amdgcn_readfirstlane(min(wave + TD_WAVES * (k - PSI), PZN - 1) * 256);
        dma4(zeros, min(zb[k >= PSI ? k - PSI : 0] + (g >> 3), zw_last) * 4u, st + TD_TILE + TN * PS * 4 + at);
      }
    } else {
      // the stage's scales of this wave's row 64 wave + lane: the dword with the one
      // FP16 scale (GSM 0), the dword of its two (GSM 1), the two dwords of its four
      // (GSM 2), the four E8M0 bytes (MXFP4); then the zero-point word
      const int k = part - WLOADS - TD_XI;
      const uint32_t g = MX ? dd * 4u : GSM == 0 ? (dd * 128u) / (uint32_t)gs : dd * (2u * GSM);
      if (k < NSC) {
        const uint32_t off = MX ? sc_base + g : GSM == 0 ? ((sc_base + g) >> 1) * 4u
                                                        : (sc_base + g) * 2u + 4u * k;
        dma4(scales, off, st + TD_TILE + k * (TD_TN * 4) + (NI == 2 ? wave : (wave & 1)) * 256);
      } else {
        dma4(zeros, (zw_base + (g >> 3)) * 4u,
             st + TD_TILE + 2 * (TD_TN * 4) + (NI == 2 ? wave : (wave & 1)) * 256);
      }
    }
  };
  auto request = [&](int d, uint32_t buf) {
#pragma unroll
    for (int part = 0; part < LOADS; ++part) request_part(d, buf, part);
  };

  // this lane's rows of the two W tiles of its wave; the parity of their first
  // scale index says which half of the fetched dword is theirs
  int wrow[NI];
  uint32_t par[NI];
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    wrow[i] = wave * (32 * NI) + i * 32 + r;
    const int n = n0 + wrow[i];
    par[i] = ((uint32_t)(n < N ? n : N - 1) * (uint32_t)G) & 1u;
  }
  const bool hook = HOOK && m0 == 0;
  uint32_t mask = 0x00F0000Fu, magic = 0x54006400u;
  asm volatile("" : "+s"(mask));   // opaque: otherwise they come back as literals of two
  asm volatile("" : "+v"(magic));  // separate instructions

  u4 xv[2][MJ];           // X operands of the step in hand and of the next: [m tile]
  u4 wv[2][NI];           // packed words of the two 64-k halves: [half][n tile], word = step % 4
  u4 av[2][NI];           // expanded W operands (four packed-half registers) of the step in hand and of the next
  uint32_t sc[NI][NSC], zw[NI];  // the stage's scale dwords and zero-point word per n tile
  // what expansion needs, per [half][n tile]: -(1024 + z), -(64 + z) and the scale in
  // both halves of a register (MXFP4: the scale as a float)
  h2 cneg[2][NI], s2v[2][NI];
  float sf[2][NI];
  // Where this lane reads inside a stage buffer, worked out once: the X piece of
  // step u in m tile 0 (tile j is 8 KB further), its four words of half s2 in n tile
  // 0 (tile 1 is 2 KB further), its scale dword.  A read is then one add of the
  // buffer's offset and an immediate.
  uint32_t xoff[8], woff[2];
#pragma unroll
  for (int u = 0; u < 8; ++u) xoff[u] = TD_W_BYTES + x_at(r, 8 * (u >> 2) + 4 * h + (u & 3));
#pragma unroll
  for (int s2 = 0; s2 < 2; ++s2) woff[s2] = w_at(wrow[0], 2 * s2 + h);
  const uint32_t scoff = TD_TILE + wrow[0] * 4;
  auto read_x = [&](u4* dst, uint32_t buf, int u) {  // step u = half u/4, MFMA u%4
    const uint8_t* p = td_lds + (buf + xoff[u]);
#pragma unroll
    for (int j = 0; j < MJ; ++j) dst[j] = *(const u4*)(p + j * 8192);
  };
  auto read_w = [&](u4* dst, uint32_t buf, int s2) {
    const uint8_t* p = td_lds + (buf + woff[s2]);
#pragma unroll
    for (int i = 0; i < NI; ++i) dst[i] = *(const u4*)(p + i * 2048);
  };
  auto read_sc = [&](uint32_t buf) {
    const uint8_t* p = td_lds + (buf + scoff);
#pragma unroll
    for (int i = 0; i < NI; ++i) {
#pragma unroll
      for (int k = 0; k < NSC; ++k) sc[i][k] = *(const uint32_t*)(p + k * (TD_TN * 4) + i * 128);
      if (ASYM) zw[i] = *(const uint32_t*)(p + 2 * (TD_TN * 4) + i * 128);
    }
  };
  auto set_group = [&](int d) {
#pragma unroll
    for (int s2 = 0; s2 < 2; ++s2)
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        if constexpr (MX) {  // block 4 d + 2 s2 + h of the row
          sf[s2][i] = mx_scale((sc[i][0] >> (8 * (2 * s2 + h))) & 0xFFu);
        } else {
          uint32_t g, s16;
          if constexpr (GSM == 0) {
            g = ((uint32_t)d * 128u) / (uint32_t)gs;
            s16 = ((par[i] + g) & 1u) ? (sc[i][0] >> 16) : (sc[i][0] & 0xFFFFu);
          } else if constexpr (GSM == 1) {
            g = 2u * d + s2;
            s16 = s2 ? (sc[i][0] >> 16) : (sc[i][0] & 0xFFFFu);
          } else {
            g = 4u * d + 2 * s2 + h;
            s16 = h ? (sc[i][s2] >> 16) : (sc[i][s2] & 0xFFFFu);
          }
          s2v[s2][i] = splat_bits(s16);
          const uint32_t z = ASYM ? ((zw[i] >> (4 * (g & 7))) & 0xFu) : 8u;
          cneg[s2][i] = as_h2(0xD400E400u | (z << 20) | z);
        }
      }
  };
  // ANY: parameters of a slice, the lane's 32 k of a half (four words, which begin in any place of a group).  The runs
  // of scales and of zero-points that begin with the first word's group come as whole dwords and are moved
  // to the bottom of their registers: sw holds two scales (gsm 4: four; MXFP4: bytes), zr the zero-points.  A word picks its
  // own by a selector of bytes and a shift.  (A wave's tiles of W are 32 rows apart, an even number of
  // scales: one place for all of them.)
  constexpr int NSL = ANY && GSM == 4 ? 3 : 2;  // scale dwords read for a slice
  [[maybe_unused]] const uint32_t gsw = (uint32_t)gs >> 3;
  [[maybe_unused]] const uint32_t row_sc = (uint32_t)(n0 + wrow[0] < N ? n0 + wrow[0] : N - 1) * (uint32_t)G;
  [[maybe_unused]] uint32_t p_sc, p_sh, p_zw, p_zs;  // where the runs lie, and their place in the first dword
  [[maybe_unused]] uint32_t rs[NI][NSL], rz[NI][2], sw[2][NI][2], zr[2][NI], rem[2];
  [[maybe_unused]] int dup[2];  // words of the half, from the lane's first on, that the stage before has
  [[maybe_unused]] uint32_t sel = 0, zsh = 0;  // of the word in hand
  [[maybe_unused]] auto slice_at = [&](int d, uint32_t buf, int s2) {
    const uint32_t wd = first_k(d) >> 3, wa = wd + 8 * s2, g0 = group_of_word(wd);
    const uint32_t ga = group_of_word(wa), gb = group_of_word(wa + 4);
    const uint32_t g = h ? gb : ga;
    const uint32_t per = MX ? 4u : gsw, ra = wa - ga * per, rb = wa + 4 - gb * per;
    rem[s2] = h ? rb : ra;
    dup[s2] = (d == stages - 1 ? (int)overlap : 0) - 8 * s2 - 4 * h;
    const uint32_t at = g - g0 + ((row_sc + g0) & (MX ? 3u : 1u)), base = buf + TD_TILE;
    p_sc = base + wrow[0] * SROW + (at >> (MX ? 2 : 1)) * SDW;
    p_sh = MX ? (at & 3) * 8 : (at & 1) * 16;
    if (ASYM) {
      p_zw = base + TN * PS * 4 + wrow[0] * ZROW + ((g >> 3) - (g0 >> 3)) * ZDW;
      p_zs = (g & 7) * 4;
    }
  };
  [[maybe_unused]] auto slice_read = [&]() {
#pragma unroll
    for (int i = 0; i < NI; ++i) {
#pragma unroll
      for (int e = 0; e < NSL; ++e) rs[i][e] = *(const uint32_t*)(td_lds + p_sc + e * SDW + i * (32 * SROW));
#pragma unroll
      for (int e = 0; e < 2; ++e)
        if (ASYM) rz[i][e] = *(const uint32_t*)(td_lds + p_zw + e * ZDW + i * (32 * ZROW));
    }
  };
  [[maybe_unused]] auto slice_set = [&](int s2) {
    // (K a multiple of 32: the words that the last stage shares with the one before it are whole slices)
    const bool none = KT == 1 && dup[s2] > 0;
#pragma unroll
    for (int i = 0; i < NI; ++i) {
#pragma unroll
      for (int e = 0; e + 1 < NSL; ++e) {
        const uint32_t run = __builtin_amdgcn_alignbit(rs[i][e + 1], rs[i][e], p_sh);
        sw[s2][i][e] = none ? 0u : run;
      }
      if (ASYM) zr[s2][i] = __builtin_amdgcn_alignbit(rz[i][1], rz[i][0], p_zs);
    }
  };
  [[maybe_unused]] auto word_at = [&](int u) {
    const int s2 = u >> 2, j = u & 3;
    if constexpr (MX) {  // the byte goes to the top of the register
      sel = KT == 2 && rem[s2] + j >= 4 ? 0x010c0c0cu : 0x000c0c0cu;
    } else if constexpr (GSM == 3) {
      const bool second = j > 0 && rem[s2] + j >= gsw;
      sel = second ? 0x03020302u : 0x01000100u;
      zsh = second ? 4u : 0u;
    } else {
      const uint32_t a = rem[s2] + j;
      sel = 0x01000100u, zsh = 0u;
      if (j > 0) sel = a >= gsw ? 0x03020302u : sel, zsh = a >= gsw ? 4u : zsh;
      if (j > 1) sel = a >= 2 * gsw ? 0x05040504u : sel, zsh = a >= 2 * gsw ? 8u : zsh;
      if (j > 2) sel = a >= 3 * gsw ? 0x07060706u : sel, zsh = a >= 3 * gsw ? 12u : zsh;
    }
    if constexpr (KT == 2) sel = j < dup[s2] ? 0x0c0c0c0cu : sel;  // (0x0c selects a byte of zeros)
  };
  [[maybe_unused]] auto word_set = [&](int u, int i) {  // (into the place of the half that step u belongs to)
    const int s2 = u >> 2;
    const uint32_t sv = __builtin_amdgcn_perm(sw[s2][i][GSM == 4 ? 1 : 0], sw[s2][i][0], sel);
    if constexpr (MX) {
      sf[s2][i] = __builtin_bit_cast(float, sv >> 1);
    } else {
      s2v[s2][i] = as_h2(sv);
      const uint32_t z = ASYM ? (zr[s2][i] >> zsh) & 0xFu : 8u;
      cneg[s2][i] = as_h2(0xD400E400u + z * 0x00100001u);
    }
  };
  // stage d lies at b, the next at bn: a slice's places are worked out ahead of the step that reads them, its runs
  // moved into place a step later (a stage's first slice: all behind the barrier that its data need)
  [[maybe_unused]] auto slice_step = [&](int d, uint32_t b, uint32_t bn, int u) {
    if (u == 0) slice_at(d, b, 1);
    if (u == 2) slice_set(1);
    if (u == 5) slice_at(d + 1, bn, 0);
  };
  // What has to be put right in a stage that has landed, by the set that holds it; then all meet.  The activations that
  // the last stage shares with the one before it are cleared; where the scales of the matrix end inside a
  // dword, which is not loaded, they are written into the last row's run.
  const bool torn = ANY && ((uint32_t)N * (uint32_t)G & (MX ? 3u : 1u)) != 0 && n0 + TN >= N;
  [[maybe_unused]] auto mend = [&](int d, uint32_t buf) {
    if (d == stages - 1)
      for (int e = wave * 64 + lane; e < TM * 16; e += TD_THREADS)
        if ((uint32_t)(e & 15) < overlap) *(u4*)(td_lds + buf + TD_W_BYTES + x_at(e >> 4, e & 15)) = u4{0u, 0u, 0u, 0u};
    if (torn && wave == 0) {
      const uint32_t per = MX ? 4u : 2u, total = (uint32_t)N * (uint32_t)G, row0 = total - (uint32_t)G;
      const uint32_t g0 = group_of_word(first_k(d) >> 3), first = total & ~(per - 1);
      const uint32_t place = (first >> (MX ? 2 : 1)) - ((row0 + g0) >> (MX ? 2 : 1));  // the dword, in the last row's run
      if (first + lane < total && place < (uint32_t)PS) {
        uint8_t* const p = td_lds + buf + TD_TILE + (N - 1 - n0) * SROW + place * SDW;
        if (MX) p[lane] = ((const uint8_t*)scales)[first + lane];
        else *(uint16_t*)p = ((const uint16_t*)scales)[first];
      }
    }
    __syncthreads();
  };
  auto hook_store = [&](const u4* src, int d, int u, int i) {
    if (HOOK && hook && d < stages && n0 + wrow[i] < N) {
      if (ANY && (u & 3) < dup[u >> 2]) return;  // (the stage before has stored it)
      *(u4*)(w_out + (size_t)(n0 + wrow[i]) * K + (ANY ? first_k(d) : d * 128u) + (u >> 2) * 64 + h * 32 + (u & 3) * 8) = src[i];
    }
  };
  auto expand = [&](u4* dst, int d, int u) {
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      if constexpr (MX) {
        h2 n4[4];
        dq_mx(wv[u >> 2][i][u & 3], sf[u >> 2][i], n4);
        dst[i] = u4{as_u32(n4[0]), as_u32(n4[1]), as_u32(n4[2]), as_u32(n4[3])};
      } else {
        dst[i] = __builtin_bit_cast(
            u4, expand_word(wv[u >> 2][i][u & 3], cneg[u >> 2][i], s2v[u >> 2][i], mask, magic));
      }
      hook_store(dst, d, u, i);
    }
  };
  // The same in four phases over the registers e0 .. e0 + nr - 1 of n tile i, one phase per
  // MFMA: the four instructions of a register depend on each other, and a wave that issues
  // them back to back waits out each one's latency.  t: the values in between.
  auto expand_phase = [&](int ph, u4* dst, uint32_t* t, int u, int i, int e0, int nr) {
    const uint32_t w = wv[u >> 2][i][u & 3];
#pragma unroll
    for (int q = 0; q < nr; ++q) {
      const int e = e0 + q;
      if constexpr (MX) {
        const float sc_f = sf[u >> 2][i];
        if (ph == q % 4)
          dst[i][e] = as_u32(e == 0   ? __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, sc_f, 0)
                             : e == 1 ? __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, sc_f, 1)
                             : e == 2 ? __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, sc_f, 2)
                                      : __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, sc_f, 3));
      } else {
        if (ph == 0) t[q] = __builtin_amdgcn_perm(0u, w, 0x0c000c00u | (uint32_t)(e << 16) | (uint32_t)e);
        if (ph == 1) t[q] = (t[q] & mask) | magic;
        if (ph == 2) t[q] = as_u32(as_h2(t[q]) + cneg[u >> 2][i]);
        if (ph == 3) dst[i][e] = as_u32(as_h2(t[q]) * s2v[u >> 2][i]);
      }
    }
  };

  f16v acc[NI][MJ];
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < MJ; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

  // Stage d + 2 is requested in pieces from step 7 of stage d - 1 (when the barrier
  // there has freed its buffer) to step 6 of stage d.  b0, b1, b2: byte offsets of
  // the buffers of stages d, d + 1, d + 2 (d + 3 takes b0 again).
  const uint32_t set_base = grp * (TD_STAGES * TD_STAGE);
  uint32_t b0 = set_base, b1 = set_base + TD_STAGE, b2 = set_base + 2 * TD_STAGE;
  request(d_first, b0);
  request(d_first + 1, b1);
#pragma unroll
  for (int part = 0; part < PPS; ++part) request_part(d_first + 2, b2, part);
  __builtin_amdgcn_s_waitcnt(waitcnt_vm(LOADS + PPS));  // stage 0 has landed
  __syncthreads();
  // (the last stage's place in its set, in sets of per_set stages each)
  [[maybe_unused]] const int last_it = (stages - 1) % per_set;
  if (ANY && (torn || (overlap && last_it == 0))) mend(d_first, b0);
  if constexpr (ANY) {
    slice_at(d_first, b0, 0);
    slice_read();
  }
  read_x(xv[0], b0, 0);
  read_w(wv[0], b0, 0);
  if constexpr (ANY) {
    slice_set(0);
    word_at(0);
#pragma unroll
    for (int i = 0; i < NI; ++i) word_set(0, i);
  } else {
    read_sc(b0);
    set_group(d_first);
  }
  expand(av[0], d_first, 0);
  [[maybe_unused]] f16v acc_first[HOOK ? NI : 1][HOOK ? MJ : 1];
#pragma unroll 1
  for (int it = 0; it < per_set; ++it) {
    const int d = d_first + it;
    if constexpr (HOOK) {
      if (d == split_at) {  // what the second set of waves of the unhooked kernel starts with
#pragma unroll
        for (int i = 0; i < NI; ++i)
#pragma unroll
          for (int j = 0; j < MJ; ++j) {
            acc_first[i][j] = acc[i][j];
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
          }
      }
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      if (u == 7) {
        // every LDS read of stage d has been issued (the X operands of step 7 during
        // step 6): once all waves are here its buffer can take stage d + 3, and stage
        // d + 1 has landed for everyone (outstanding: all of stage d + 2)
        __builtin_amdgcn_s_waitcnt(waitcnt_vm(LOADS));
        __syncthreads();
        if (ANY && (torn || (overlap && it + 1 == last_it))) mend(d + 1, b1);
#pragma unroll
        for (int part = 0; part < PPS; ++part) request_part(d + 3, b0, part);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (ANY) slice_read();
        read_x(xv[0], b1, 0);
        read_w(wv[0], b1, 0);
        if constexpr (ANY) {
          slice_set(0);
          word_at(0);
#pragma unroll
          for (int i = 0; i < NI; ++i) word_set(0, i);
        } else {
          read_sc(b1);
          set_group(d + 1);
        }
        expand(av[0], d + 1, 0);
      } else {
#pragma unroll
        for (int i = 0; i < PPS; ++i)
          if (PPS * (u + 1) + i < LOADS) request_part(d + 2, b2, PPS * (u + 1) + i);
        __builtin_amdgcn_sched_barrier(0);
        if (ANY && u == 1) slice_read();
        read_x(xv[(u + 1) & 1], b0, u + 1);
        if (u == 0) read_w(wv[1], b0, 1);
        if constexpr (!PHASED) {
          if constexpr (ANY) {
            slice_step(d, b0, b1, u);
            word_at(u + 1);
#pragma unroll
            for (int i = 0; i < NI; ++i) word_set(u + 1, i);
          }
          expand(av[(u + 1) & 1], d, u + 1);
        }
      }
      constexpr int NM = NI * MJ;  // MFMAs of a step
      auto mfma = [&](int k) {
        const int i = k / MJ, j = k % MJ;
        if (KG == 1 || d < stages)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(
              __builtin_bit_cast(h8, av[u & 1][i]), __builtin_bit_cast(h8, xv[u & 1][j]), acc[i][j], 0, 0, 0);
      };
      bool done = false;
      if constexpr (PHASED) if (u < 7) {
        done = true;
        // the operands of step u + 1, expanded under this step's MFMAs: four MFMAs per group
        // of RPG registers, one phase under each
        constexpr int RPG = 16 * NI / NM;  // registers per group of four MFMAs
        uint32_t tmp[RPG];
#pragma unroll
        for (int k = 0; k < NM; ++k) {
          if constexpr (ANY) {  // ahead of the phase that takes them; then the next step's places
            if (k == 0) word_at(u + 1);
            if (RPG == 4 ? (k & 3) == 0 : k == 0) {
              word_set(u + 1, RPG == 4 ? k >> 2 : 0);
              if (RPG == 8) word_set(u + 1, 1);
            }
            if (k == NM - 1) slice_step(d, b0, b1, u);
          }
          if constexpr (RPG == 4) {  // a group of four MFMAs per word
            expand_phase(k & 3, av[(u + 1) & 1], tmp, u + 1, k >> 2, 0, 4);
            if ((k & 3) == 3) hook_store(av[(u + 1) & 1], d, u + 1, k >> 2);
          } else {  // four MFMAs in all: both words under them
            static_assert(RPG == 8 && NI == 2, "64 rows of X against two tiles of W");
            expand_phase(k & 3, av[(u + 1) & 1], tmp, u + 1, 0, 0, 4);
            expand_phase(k & 3, av[(u + 1) & 1], tmp + 4, u + 1, 1, 0, 4);
            if ((k & 3) == 3) {
              hook_store(av[(u + 1) & 1], d, u + 1, 0);
              hook_store(av[(u + 1) & 1], d, u + 1, 1);
            }
          }
          mfma(k);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      if (!done) {
#pragma unroll
      for (int k = 0; k < NM; ++k) mfma(k);
      if constexpr (!ANY) {
      // LDS reads first, then the expansion spread evenly under the MFMAs: a wave
      // can issue about six vector instructions in the shadow of one MFMA
      // vector instructions of a step (16 per word, a few more), shared out over its MFMAs
      constexpr int VPM = (16 * NI + 8 + NM - 1) / NM, VPM0 = VPM + 2;
      constexpr int VPM7 = (16 * NI + 16 + NM / 2) / (NM / 2 + 1);
      if (u == 7) {
        // the words to expand have only just been asked for: the first MFMAs cover that
        __builtin_amdgcn_sched_group_barrier(0x100, NI + MJ + NI * NSC + (ASYM ? NI : 0), 0);
#pragma unroll
        for (int k = 0; k < NM / 2 - 1; ++k) __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
#pragma unroll
        for (int k = 0; k < NM / 2 + 1; ++k) {
          __builtin_amdgcn_sched_group_barrier(0x002, VPM7, 0);
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        }
      } else {
        if (u == 0) __builtin_amdgcn_sched_group_barrier(0x100, MJ + NI, 0);
        else __builtin_amdgcn_sched_group_barrier(0x100, MJ, 0);
#pragma unroll
        for (int k = 0; k < NM; ++k) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          if (u == 0) __builtin_amdgcn_sched_group_barrier(0x002, VPM0, 0);
          else __builtin_amdgcn_sched_group_barrier(0x002, VPM, 0);
        }
      }
      }
      __builtin_amdgcn_sched_barrier(0);
      }
    }
    const uint32_t first = b0;
    b0 = b1;
    b1 = b2;
    b2 = first;
  }
  __builtin_amdgcn_s_waitcnt(waitcnt_vm(0));  // nothing may still be writing LDS at exit
  if constexpr (HOOK) {
    if (split_at < stages) {
#pragma unroll
      for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int j = 0; j < MJ; ++j) acc[i][j] = acc_first[i][j] + acc[i][j];
    }
  }
  if constexpr (KG == 2) {
    // the second set's sums go to the first through LDS (the stage buffers are free once
    // every wave is here): first set + second set, in that order
    __syncthreads();
    float* mine = (float*)td_lds + (size_t)wave * (NI * MJ * 16 * 64);
    if (grp == 1) {
#pragma unroll
      for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int j = 0; j < MJ; ++j)
#pragma unroll
          for (int e = 0; e < 16; ++e) mine[((i * MJ + j) * 16 + e) * 64 + lane] = acc[i][j][e];
    }
    __syncthreads();
    if (grp == 1) return;
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
      for (int j = 0; j < MJ; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[i][j][e] += mine[((i * MJ + j) * 16 + e) * 64 + lane];
  }

  // A lane holds, of each 32 x 32 tile, n = 8 q + 4 h + e for m = tile row r.  Whole
  // tiles go through LDS (free by now) so that every store instruction writes eight
  // whole 128-byte lines instead of 16 bytes of each of 32: a wave lays its 128 (m)
  // x 64 (n) block out in rows of 144 bytes and reads it back 16 bytes a lane.
  const bool whole = m0 + TD_TM <= M && n0 + TD_TN <= N && (N & 7) == 0 && ((uintptr_t)c & 15) == 0;
  if (whole) {
    constexpr int RB = 64 * NI, PITCH = RB + 16;  // bytes of a row of the wave's block, and its LDS pitch
    constexpr int PP = RB / 16, ROWS = 64 / PP;   // 16-byte pieces per row, rows per store instruction
    __syncthreads();  // no wave reads a stage buffer any more, no load is landing in one
    uint8_t* mine = td_lds + wave * (TD_TM * PITCH);
#pragma unroll
    for (int j = 0; j < MJ; ++j)
#pragma unroll
      for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          h4 out;
#pragma unroll
          for (int e = 0; e < 4; ++e) out[e] = (_Float16)acc[i][j][4 * q + e];
          *(h4*)(mine + (j * 32 + r) * PITCH + i * 64 + q * 16 + h * 8) = out;
        }
    w4_half* cw = c + (size_t)m0 * N + n0 + wave * (32 * NI);
#pragma unroll
    for (int it = 0; it < TD_TM / ROWS; ++it) {
      const int row = it * ROWS + lane / PP, piece = lane % PP;
      const u4 v = *(const u4*)(mine + row * PITCH + piece * 16);
      *(u4*)(cw + (size_t)row * N + piece * 8) = v;
    }
    return;
  }
#pragma unroll
  for (int j = 0; j < MJ; ++j) {
    const int m = m0 + j * 32 + r;
    if (m >= M) continue;
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int nn = n0 + wave * (32 * NI) + i * 32 + 8 * q + 4 * h;
        w4_half* dst = c + (size_t)m * N + nn;
        if (nn + 3 < N && ((uintptr_t)dst & 7) == 0) {
          h4 out;
#pragma unroll
          for (int e = 0; e < 4; ++e) out[e] = (_Float16)acc[i][j][4 * q + e];
          *(h4*)dst = out;
        } else {
          const int left = N - nn;
          if (left > 0) dst[0] = __builtin_bit_cast(uint16_t, (_Float16)acc[i][j][4 * q + 0]);
          if (left > 1) dst[1] = __builtin_bit_cast(uint16_t, (_Float16)acc[i][j][4 * q + 1]);
          if (left > 2) dst[2] = __builtin_bit_cast(uint16_t, (_Float16)acc[i][j][4 * q + 2]);
          if (left > 3) dst[3] = __builtin_bit_cast(uint16_t, (_Float16)acc[i][j][4 * q + 3]);
        }
      }
  }
}

// group_mul: of the kernels for any group, ceil(2^31 / (gs / 8)): the group of word w is (2 w group_mul) >> 32
template <int FMT, int GSM, bool HOOK, int TM, int TN, int KG = 1, int KT = 0>
hipError_t launch(const WView& v, const w4_half* x, w4_half* c, w4_half* w_out, int M,
                  hipStream_t s, int tiles_n, int tiles_m, int split_at, uint32_t group_mul = 0) {
  constexpr int TD_LDS = KG * td_lds_bytes(TM, TN, td_planes(FMT, GSM, KT)) + td_any_slack(TN, KT);
  static_assert(TD_LDS <= 160 * 1024, "the stage buffers of every set of waves fit LDS");
  // more than 64 KB of LDS has to be granted per device, once
  static std::atomic<bool> granted[64] = {};
  int dev = 0;
  if (hipError_t e = hipGetDevice(&dev); e != hipSuccess) return e;
  if (dev < 0 || dev >= 64 || !granted[dev]) {
    const hipError_t e = hipFuncSetAttribute((const void*)w4_tile_dma_kernel<FMT, GSM, HOOK, TM, TN, KG, KT>,
                                             hipFuncAttributeMaxDynamicSharedMemorySize, TD_LDS);
    if (e != hipSuccess) return e;
    if (dev >= 0 && dev < 64) granted[dev] = true;
  }
  w4_tile_dma_kernel<FMT, GSM, HOOK, TM, TN, KG, KT>
      <<<dim3((unsigned)(tiles_n * tiles_m)), dim3(TD_THREADS * KG), TD_LDS, s>>>(
          v.q, v.scales, v.zeros, x, c, w_out, v.N, v.K, v.mx ? v.B : v.G, v.gs, M, tiles_n,
          tiles_m, split_at, group_mul);
  return hipGetLastError();
}

}  // namespace
}  // namespace w4k
