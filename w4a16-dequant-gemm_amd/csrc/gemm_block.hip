// W4A16 / MXFP4 GEMM for middle M (9 to some hundred rows, at long K from 3 on): a workgroup owns a block of
// 16 NT rows of W x 16 MT activation rows, its eight waves split K.  mma.cuh:63-230 is the
// reference's kernel for this path.
//
// What bounds these shapes is the path from L2 into a compute unit: it takes 1 KB per 7 - 10 ns
// whatever lies in it, as long as the 4 (better 8) neighbouring lanes of a load instruction lie in
// one line; a load in MFMA operand layout (neighbouring lanes in different rows) takes 28 ns.  (A block
// takes 15 ns a KB with its arithmetic: MXFP4, N = 4096, M = 50 2.0 us for each further unit of 256 k of the eight
// waves, 128 KB, whether the codes come from memory or from a cache.)  So
//   * the block is as square as the operands' sizes ask for: per k a workgroup moves 8 NT bytes of codes
//     and 32 MT bytes of activations, N = 4096, M = 64: 64 B with 64 x 16 blocks against 136 with one
//     16-row tile of W per workgroup and all of x;
//   * both operands come as whole lines by global_load_lds_dwordx4 into LDS that belongs to one
//     wave, are read back into registers in operand layout (XOR-swizzled, conflict-free) and their
//     place is requested again at once, so that the whole LDS is on its way while the wave expands
//     and multiplies.  Waves meet only at the two ends: group parameters of the block's rows are
//     copied into LDS first, and the waves' sums are added in wave order last.
// Workgroups that share rows of W are neighbours on one XCD, whose L2 then gets them once.
#include <atomic>
#include <type_traits>
#include <utility>

#include "dq.cuh"
#include "kernels.h"

namespace w4k {
namespace {

// (the compiler takes lambdas this large out of line, with their registers in scratch memory)
#define BK_INLINE __attribute__((always_inline))

typedef __attribute__((address_space(3))) void* lds_ptr;
constexpr int BK_WAVES = 8, BK_THREADS = 64 * BK_WAVES;
constexpr int BK_UNIT = 256;  // k of a unit: one 128-byte line of a row of codes, two of a row of x
constexpr int BK_XS = 2;      // pieces in a wave's ring of x
constexpr uint32_t BK_GRID_Y = 65535;
constexpr int bk_wave_bytes(int NT, int XS) { return NT * 2048 + XS * 4096; }
extern __shared__ __attribute__((aligned(16))) uint8_t bk_lds[];

// f(integral_constant<int, 0>), f(integral_constant<int, 1>), ...: a loop whose index is
// a constant expression inside the body (wait counts are instruction immediates)
template <class F, int... I>
__device__ __forceinline__ void bk_for(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}

// (One wait state between the write of M0 and the load that takes its LDS address from it.)
__device__ __forceinline__ void bk_dma(uint32_t off, const void* base, uint32_t dst) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"(off), "s"(base), "s"(dst) : "memory", "m0");
}

__device__ __forceinline__ void bk_dma4(uint32_t off, const void* base, uint32_t dst) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dword %0, %1" : : "v"(off), "s"(base), "s"(dst) : "memory", "m0");
}

// FMT: 0 W4 symmetric, 1 W4 with zero-points, 2 MXFP4.  G: groups (W4) or blocks (MXFP4) per row.
// group_mul: ceil(2^31 / (gs / 8)): the group of word w is (2 w group_mul) >> 32.  XS: pieces of x (16 rows x 128 k, 4 KB) in a
// wave's ring; three measured no better than two.  LATE (W4, gs a multiple of 128: a chunk of 128 k is in one
// group): the operands are the codes minus the zero-point, exact in FP16, and the scale is applied to a
// chunk's FP32 sums, as the resident kernel does in the shapes that this one took over from it
// (rounding q s to FP16 first: 2.7e-4 from the product in FP64 instead of 2.1e-4, K = 4096, M = 16).
// GM (W4 with groups that a lane's 32 k of a chunk do not all belong to one of): 1 groups of 32 or more k, at most two
// of which meet in such a slice, 2 smaller ones, at most four.  A slice's runs of scales and zero-points come as
// whole dwords and are moved to the bottom of their registers, from which a word picks its own by a
// selector of bytes and a shift.  RAG: K is no multiple of 32 (rows of codes are 4-byte aligned only) or N none of 16: codes
// come dword by dword.  window (GM = 2): at long K the parameters of small groups are more than LDS holds (gs = 8, K = 11008: 3.4 KB
// a row), and the block has those of this many units of every wave at a time, copied while all waves wait (K = 11008, gs = 8,
// N = 4096, M = 99: 32 x 64 blocks 34 us; 16 x 16 ones, whose parameters fit, and 32 x 128 tiles 79).
template <int FMT, int NT, int MT, int XS, bool AHEAD, bool LATE, int GM, bool RAG>
__global__ __launch_bounds__(BK_THREADS) void mfma_block_kernel(
    const uint32_t* __restrict__ q, const void* __restrict__ scales, const uint32_t* __restrict__ zeros,
    const w4_half* __restrict__ x, w4_half* __restrict__ c, const int N, const int K, const int M, const int G,
    const int gs, const uint32_t group_mul, const int window, w4_half* __restrict__ w_out) {
  constexpr bool MX = FMT == 2;
  static_assert(!(MX && LATE), "an MXFP4 chunk has four scales");
  static_assert(GM == 0 || (!MX && !LATE), "scales of a chunk or of MXFP4 blocks need no selector");
  constexpr int CL = RAG ? 8 * NT : 2 * NT;  // load instructions of a unit's codes
  constexpr int WB = bk_wave_bytes(NT, XS), ROWS = 16 * NT, NP = 2 * MT;
  // Step of a unit at which its codes have been read back and the next unit's are requested: with
  // many row tiles one chunk's codes are read at a time (registers).
  constexpr int PC = !AHEAD && MT >= 3 ? MT : 0;
  static_assert(XS >= 2 && XS <= (PC ? MT : NP), "a unit's first piece is requested after its codes");
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, b = lane >> 4;
  // x: XCD + 8 x block along M, y (and z, from 65535 on): eight blocks along N.  (As one number, whose division by a count
  // in memory came before the first request, a call took 0.2 us longer.  The arguments up to G are in registers when a wave
  // starts.)
  const uint32_t first_n = ((blockIdx.x & 7) + 8 * (blockIdx.y + BK_GRID_Y * blockIdx.z)) * ROWS;
  if (first_n >= (uint32_t)N) return;
  const int n0 = (int)first_n, m0 = (int)(blockIdx.x >> 3) * (16 * MT);
  const int units = (K + BK_UNIT - 1) / BK_UNIT;
  const uint32_t wrow = (uint32_t)(K >> 1), xrow = (uint32_t)(K * 2);
  const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_ptr)bk_lds;
  const uint32_t region = lds0 + (uint32_t)wave * WB;
  uint8_t* const mine = bk_lds + wave * WB;
  uint8_t* const params = bk_lds + BK_WAVES * WB;

  // ---- group parameters of the block's rows: one contiguous run each, 1 KB a load ----
  const int live = min(ROWS, N - n0);
  [[maybe_unused]] uint8_t* rest_s = nullptr;  // RAG: bytes of the matrix's last rows that are no whole 16, and their places
  [[maybe_unused]] uint8_t* rest_z = nullptr;
  [[maybe_unused]] uint8_t byte_s = 0, byte_z = 0;
  const int pb = live * G * (MX ? 1 : 2), wg = words(G), zb = live * wg * 4;
  const int units_most = (units + BK_WAVES - 1) / BK_WAVES;  // of a wave
  const bool windows = GM == 2 && window < units_most;
  const int GP = windows ? window * (BK_WAVES * BK_UNIT) / gs : G;  // groups of a row that LDS has
  const int wgp = windows ? GP >> 3 : wg;
  const int zoff = (ROWS * GP * (MX ? 1 : 2) + 1023) & ~1023;
  // the parameters of window j, a dword a lane: scales of a row in whole loads, zero-points of all rows as one run
  auto copy_window = [&](int j) BK_INLINE {
    const int left = min(GP, G - j * GP);
    for (int row = wave; row < ROWS; row += BK_WAVES) {
      const char* ps = (const char*)scales + ((size_t)(n0 + min(row, live - 1)) * G + (size_t)j * GP) * 2;
      for (int o = 0; o < GP * 2; o += 256)
        bk_dma4((uint32_t)min(o + lane * 4, left * 2 - 4), ps, lds0 + BK_WAVES * WB + row * GP * 2 + o);
    }
    if constexpr (FMT == 1) {
      const char* pz = (const char*)zeros + ((size_t)n0 * wg + (size_t)j * wgp) * 4;
      for (int o = wave * 64; o < ROWS * wgp; o += BK_WAVES * 64) {
        const int row = (o + lane) / wgp, col = (o + lane) - row * wgp;
        bk_dma4((uint32_t)(min(row, live - 1) * wg + min(col, words(left) - 1)) * 4, pz, lds0 + BK_WAVES * WB + zoff + o * 4);
      }
    }
  };
  if (windows) {
    copy_window(0);
  } else {
    const char* ps = (const char*)scales + (size_t)n0 * G * (MX ? 1 : 2);
    const int pw = RAG ? pb & ~15 : pb, zw16 = RAG ? zb & ~15 : zb;  // (16 rows have whole pieces of 16 bytes)
    for (int o = wave * 1024; o < pw; o += BK_WAVES * 1024)
      bk_dma((uint32_t)min(o + lane * 16, pw - 16), ps, lds0 + BK_WAVES * WB + o);
    const char* pz = FMT == 1 ? (const char*)zeros + (size_t)n0 * wg * 4 : nullptr;
    if constexpr (RAG) {
      // (written by the wave whose load ends there, once it has landed: its lanes past the end write behind it)
      if (lane < (pb & 15) && wave == (max(pw - 1, 0) >> 10) % BK_WAVES) {
        rest_s = params + pw + lane;
        byte_s = (uint8_t)ps[pw + lane];
      }
      if (FMT == 1 && lane < (zb & 15) && wave == (max(zw16 - 1, 0) >> 10) % BK_WAVES) {
        rest_z = params + zoff + zw16 + lane;
        byte_z = (uint8_t)pz[zw16 + lane];
      }
    }
    if (FMT == 1) {
      for (int o = wave * 1024; o < zw16; o += BK_WAVES * 1024)
        bk_dma((uint32_t)min(o + lane * 16, zw16 - 16), pz, lds0 + BK_WAVES * WB + zoff + o);
    }
  }

  // ---- requests ----
  // codes of a unit: 2 NT loads of 8 rows x 128 bytes; lane l: row l / 8, piece (l % 8) ^ key, key = (row of the
  // tile / 2) % 8, so that the 16 rows a piece is read back from lie in 16 distinct groups of banks.  A tile past
  // N (whole ones: N is a multiple of 16) repeats the block's first.
  // (In both requests the pieces past the end of a row, which only the last unit has, are a branch of
  // their own: as selects they were a third of the loop's vector instructions.)
  uint32_t cpiece[2], coff[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int row = 8 * h + (lane >> 3);
    cpiece[h] = (uint32_t)(((lane & 7) ^ (row >> 1)) & 7) * 16;
    coff[h] = (uint32_t)row * wrow + cpiece[h];
  }
  const char* const qb = (const char*)q + (size_t)n0 * wrow;
  auto request_codes = [&](int U) BK_INLINE {
    const bool tail = (U + 1) * BK_UNIT > K;
    if constexpr (RAG) {  // two rows a load, a dword a lane, to the places that the 16-byte loads give them
      int lr = lane;
      asm volatile("" : "+v"(lr) : : "memory");  // (offsets ahead of the loop would take registers)
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int row = 2 * e + (lr >> 5);
        const uint32_t in = (uint32_t)((((lr & 31) >> 2) ^ e) * 16 + (lr & 3) * 4);
        uint32_t o = in;
        if (tail) {
          if ((uint32_t)U * 128 + in >= wrow) o = 0;
          asm volatile("" : "+v"(o) : : "memory");
        }
        const uint32_t own = o + (uint32_t)row * wrow;
#pragma unroll
        for (int t = 0; t < NT; ++t) {
          const int first = 16 * t < live ? 16 * t : 0;
          uint32_t ot = own;
          if (first + 16 > live) {  // rows past N repeat the last one
            ot = o + (uint32_t)min(row, live - 1 - first) * wrow;
            asm volatile("" : "+v"(ot) : : "memory");
          }
          bk_dma4(ot, qb + (size_t)first * wrow + (size_t)U * 128, region + t * 2048u + e * 256u);
        }
      }
      return;
    }
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const char* base = qb + (16 * t < live ? (size_t)(16 * t) * wrow : 0) + (size_t)U * 128;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        uint32_t o = coff[h];
        if (tail) {  // the unit's first piece instead
          if ((uint32_t)U * 128 + cpiece[h] >= wrow) o -= cpiece[h];
          asm volatile("" : "+v"(o) : : "memory");
        }
        bk_dma(o, base, region + (2 * t + h) * 1024u);
      }
    }
  };
  // piece p = (chunk p / MT of the unit, row tile p % MT): 4 loads of 4 rows x 256 bytes, piece (l % 16) ^ (row % 16)
  const char* const xb = (const char*)x + (size_t)m0 * xrow;
  const int mlast = M - 1 - m0;
  // Offsets are worked out once: for every tile and load where registers allow; larger blocks have those of a whole
  // tile of rows, from its first row, and of the tile that M ends in, which stands in for the tiles
  // behind it as well.
  constexpr bool XALL = MT <= 4;
  const int mend = mlast >> 4;
  uint32_t xoff[XALL ? MT : 2][4];
#pragma unroll
  for (int i = 0; i < (XALL ? MT : 2); ++i)
#pragma unroll
    for (int rq = 0; rq < 4; ++rq) {
      const int r16 = 4 * rq + (lane >> 4), row = XALL ? min(16 * i + r16, mlast) : i ? min(16 * mend + r16, mlast) : r16;
      xoff[i][rq] = (uint32_t)row * xrow + (uint32_t)(((lane & 15) ^ r16) * 16);
    }
  auto request_x = [&](int U, int p, int slot) BK_INLINE {
    const int ch = p / MT, mt = p % MT;
    const uint32_t k2 = (uint32_t)(U * 2 + ch) * 256u;  // byte of the row
    const uint32_t dst = region + NT * 2048u + (uint32_t)slot * 4096u;
    const char* const tile = xb + (!XALL && mt < mend ? (size_t)(16 * mt) * xrow : 0);
    auto offset = [&](int rq) BK_INLINE { return XALL ? xoff[mt][rq] : mt < mend ? xoff[0][rq] : xoff[1][rq]; };
    if (k2 + 256 > xrow) {
      asm volatile("" ::: "memory");
      const bool past = k2 >= xrow;  // all of the chunk: the chunk before instead
      const char* base = tile + (past ? k2 - 256 : k2);
#pragma unroll
      for (int rq = 0; rq < 4; ++rq) {
        const uint32_t piece = (uint32_t)(((lane & 15) ^ (4 * rq + (lane >> 4))) * 16);
        bk_dma(offset(rq) - (past || k2 + piece >= xrow ? piece : 0u), base, dst + rq * 1024u);
      }
    } else {
      const char* base = tile + k2;
#pragma unroll
      for (int rq = 0; rq < 4; ++rq) bk_dma(offset(rq), base, dst + rq * 1024u);
    }
  };

  const int nu = (units - wave + BK_WAVES - 1) / BK_WAVES;  // wave w takes units w, w + 8, ...
  if (nu > 0) {
    request_codes(wave);
#pragma unroll
    for (int p = 0; p < XS; ++p) request_x(wave, p, p);
    __builtin_amdgcn_s_waitcnt(waitcnt_vm(CL + 4 * XS));
  } else {
    __builtin_amdgcn_s_waitcnt(waitcnt_vm(0));
  }
  if constexpr (RAG) {
    if (rest_s) *rest_s = byte_s;
    if (rest_z) *rest_z = byte_z;
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
  }
  asm volatile("s_barrier" ::: "memory");  // the parameters are there

  uint32_t mask = 0x00F0000Fu, magic = 0x54006400u;
  asm volatile("" : "+s"(mask));   // opaque: as literals they cost two instructions
  asm volatile("" : "+v"(magic));  // instead of one and-or
  f4 acc[NT][MT];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[t][mt] = f4{0.f, 0.f, 0.f, 0.f};
  u4 cw[PC ? 1 : 2][NT];
  h8 A[NT][4];
  // group parameters of a lane's 32 k of a chunk, and their group; LATE: scales of the rows of its four sums
  struct runs_t {  // GM: dwords that hold the slice's scales
    uint32_t d[GM == 2 ? 3 : 2];
  };
  typedef std::conditional_t<LATE, h4, std::conditional_t<(GM > 0), runs_t, uint32_t>> scale_t;
  typedef std::conditional_t<(GM > 0), u2, uint32_t> zero_t;
  scale_t sc[NT];
  zero_t zw[NT];
  [[maybe_unused]] const int gsw = gs >> 3;
  [[maybe_unused]] h4 late[NT];  // the scales of the chunk that is multiplied
  int g = 0, slot = 0;  // slot: of the piece that is multiplied
  [[maybe_unused]] int g_first = 0, done = 0;  // the window's first group; units that the wave has begun
  const bool hook = w_out && m0 == 0;

  auto read_codes = [&](int h, u4* w) BK_INLINE {
#pragma unroll
    for (int t = 0; t < NT; ++t)
      w[t] = *(const u4*)(mine + t * 2048 + r * 128 + (((4 * h + b) ^ (r >> 1)) & 7) * 16);
  };
  auto read_x = [&](int at, h8* v) BK_INLINE {  // B operands: MFMA j contracts k = 128 chunk + 32 b + 8 j .. + 7 = piece 4 b + j
#pragma unroll
    for (int j = 0; j < 4; ++j)
      v[j] = *(const h8*)(mine + NT * 2048 + at * 4096 + (r >> 2) * 1024 + ((r & 3) * 16 + ((4 * b + j) ^ r)) * 16);
  };
  auto read_params = [&](int chunk) BK_INLINE {
    const int kc = min(chunk * 128 + (LATE ? 0 : 32 * b), RAG ? K - 8 : K - 32);
    g = MX ? (kc >> 5) : (int)__umulhi((uint32_t)kc >> 2, group_mul);
    if constexpr (GM > 0) {
      const int gw = GM == 2 ? g - g_first : g, pitch = GM == 2 ? GP : G, zpitch = GM == 2 ? wgp : wg;
      const uint8_t* ps = params + ((r * pitch + gw) >> 1) * 4;
      const uint8_t* pz = params + zoff + (r * zpitch + (gw >> 3)) * 4;
#pragma unroll
      for (int t = 0; t < NT; ++t) {
#pragma unroll
        for (int e = 0; e < (GM == 2 ? 3 : 2); ++e) sc[t].d[e] = *(const uint32_t*)(ps + t * 32 * pitch + e * 4);
        if (FMT == 1) zw[t] = u2{*(const uint32_t*)(pz + t * 64 * zpitch), *(const uint32_t*)(pz + t * 64 * zpitch + 4)};
      }
      return;
    }
    if constexpr (GM == 0) {
      const uint8_t* ps = params + ((LATE ? 4 * b : r) * G + g) * (MX ? 1 : 2);
      const uint8_t* pz = params + zoff + (r * wg + (g >> 3)) * 4;
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        if constexpr (LATE) {
          const _Float16* p = (const _Float16*)ps + t * 16 * G;
          sc[t] = h4{p[0], p[G], p[2 * G], p[3 * G]};
        } else {
          sc[t] = MX ? ps[t * 16 * G] : *(const uint16_t*)(ps + t * 32 * G);
        }
        if (FMT == 1) zw[t] = *(const uint32_t*)(pz + t * 64 * wg);
      }
      // Lanes past the end of the row hold codes of another group than g's: with its scale they can overflow FP16,
      // and infinity times the zeroed activations is NaN.  A scale of 0 (MXFP4: 2^-127) makes them zeros.
      // (LATE: the codes are finite, the scale of a chunk that is past the end as a whole may not be.)
      if (chunk * 128 + 128 > K) {
        if (chunk * 128 + (LATE ? 0 : 32 * b) >= K) {
#pragma unroll
          for (int t = 0; t < NT; ++t) sc[t] = scale_t{};
        }
        asm volatile("" ::: "memory");
      }
    }
  };
  auto request_next = [&](auto pc, int U, bool more) BK_INLINE {  // into the places that are free at step p of unit U
    constexpr int p = decltype(pc)::value;
    if (p == PC && more) request_codes(U + BK_WAVES);
    if (p + XS < NP) request_x(U, p + XS, slot);
    else if (more) request_x(U + BK_WAVES, p + XS - NP, slot);
    slot = slot + 1 < XS ? slot + 1 : 0;
  };
  // the codes in w, with the parameters given, become the weights of a chunk; k: the lane's first
  auto expand = [&](const u4* w, const scale_t* scale, const zero_t* zword, int group, int k) BK_INLINE {
    if constexpr (GM > 0) {
      const int rem = (int)((uint32_t)min(k, RAG ? K - 8 : K - 32) >> 3) - group * gsw;
      uint32_t sel[4], zsh[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        sel[j] = 0x01000100u, zsh[j] = 0u;
        if (j > 0) sel[j] = rem + j >= gsw ? 0x03020302u : sel[j], zsh[j] = rem + j >= gsw ? 4u : zsh[j];
        if (GM == 2 && j > 1) sel[j] = rem + j >= 2 * gsw ? 0x05040504u : sel[j], zsh[j] = rem + j >= 2 * gsw ? 8u : zsh[j];
        if (GM == 2 && j > 2) sel[j] = rem + j >= 3 * gsw ? 0x07060706u : sel[j], zsh[j] = rem + j >= 3 * gsw ? 12u : zsh[j];
      }
      if ((k & ~127) + 128 > K) {  // words past the end of the row: zeros, whatever scale they would have
#pragma unroll
        for (int j = 0; j < 4; ++j) sel[j] = k + 8 * j >= K ? 0x0c0c0c0cu : sel[j];
        asm volatile("" ::: "memory");
      }
      const uint32_t odd = ((uint32_t)(r * G + group) & 1u) * 16u;
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const uint32_t lo = __builtin_amdgcn_alignbit(scale[t].d[1], scale[t].d[0], odd);
        uint32_t hi = lo, zr = 0;
        if constexpr (GM == 2) hi = __builtin_amdgcn_alignbit(scale[t].d[2], scale[t].d[1], odd);
        if constexpr (FMT == 1) zr = __builtin_amdgcn_alignbit(zword[t][1], zword[t][0], 4 * (group & 7));
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const uint32_t z = FMT == 1 ? (zr >> zsh[j]) & 0xFu : 8u;
          const h2 cneg = as_h2(0xD400E400u + z * 0x00100001u), s2 = as_h2(__builtin_amdgcn_perm(hi, lo, sel[j]));
          A[t][j] = expand_word(w[t][j], cneg, s2, mask, magic);
        }
      }
    } else {
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        h2 cneg, s2 = h2{0, 0};
        float sf = 0.f;
        if constexpr (MX) {
          sf = mx_scale(scale[t]);
        } else {
          const uint32_t z = FMT == 1 ? ((zword[t] >> (4 * (group & 7))) & 0xFu) : 8u;
          cneg = as_h2(0xD400E400u | (z << 20) | z);
          if constexpr (LATE) late[t] = scale[t];
          else s2 = splat_bits(scale[t]);
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          if (MX) {
            h2 n4[4];
            dq_mx(w[t][j], sf, n4);
            A[t][j] = __builtin_bit_cast(h8, u4{as_u32(n4[0]), as_u32(n4[1]), as_u32(n4[2]), as_u32(n4[3])});
          } else {
            A[t][j] = expand_word<!LATE>(w[t][j], cneg, s2, mask, magic);
          }
        }
      }
    }
    if constexpr (RAG && MX) {  // (a scale may overflow the codes of a slice that the row ends in)
      if ((k & ~127) + 128 > K) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (k + 8 * j >= K) {
#pragma unroll
            for (int t = 0; t < NT; ++t) A[t][j] = __builtin_bit_cast(h8, u4{0u, 0u, 0u, 0u});
          }
        asm volatile("" ::: "memory");
      }
    }
    if (hook) {  // these registers are the weights (LATE: times the scale of the lane's row)
      int row = r;
      asm volatile("" : "+v"(row) : : "memory");  // (addresses ahead of the loop would take registers in every call)
#pragma unroll
      for (int t = 0; t < NT; ++t)
        if (16 * t + (RAG ? row : 0) < live && k < K) {
          const _Float16 own = LATE ? *(const _Float16*)(params + ((t * 16 + row) * G + group) * 2) : (_Float16)1.f;
#pragma unroll
          for (int j = 0; j < 4; ++j)
            if (!RAG || k + 8 * j < K)
              *(h8*)(w_out + (size_t)(n0 + 16 * t + row) * K + k + 8 * j) = LATE ? A[t][j] * own : A[t][j];
        }
    }
  };
  // LATE: a chunk's sums of two tiles of W, which are scaled while the next two multiply
  constexpr int ST = 2, LAST = (NT - 1) / ST * ST;
  [[maybe_unused]] f4 held[ST];
  auto add_scaled = [&](int t0, int mt) BK_INLINE {
#pragma unroll
    for (int t = t0; t < t0 + ST && t < NT; ++t) {
      asm volatile("" : "+v"(late[t]));  // (stays in halves: v_fma_mix_f32 takes them)
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[t][mt][i] = fmaf(held[t - t0][i], (float)late[t][i], acc[t][mt][i]);
      // (here and not at the end of the unit, where the compiler would put it with all chunk sums alive)
      asm volatile("" : "+v"(acc[t][mt]));
    }
  };
  auto multiply = [&](auto mtc, int chunk, h8* v) BK_INLINE {
    if (chunk * 128 + 128 > K) {  // the row ends inside this chunk: activations past it are zero
      if constexpr (RAG) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (chunk * 128 + 32 * b + 8 * j >= K) v[j] = __builtin_bit_cast(h8, u4{0u, 0u, 0u, 0u});
      } else if (chunk * 128 + 32 * b >= K) {
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = __builtin_bit_cast(h8, u4{0u, 0u, 0u, 0u});
      }
      asm volatile("" ::: "memory");
    }
    if constexpr (LATE) {
      constexpr int mt = decltype(mtc)::value;
#pragma unroll
      for (int t0 = 0; t0 < NT; t0 += ST) {
        f4 part[ST];
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int t = t0; t < t0 + ST && t < NT; ++t)
            part[t - t0] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A[t][j], v[j], j ? part[t - t0] : f4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
        if (t0 > 0) add_scaled(t0 - ST, mt);
        else if (mt > 0) add_scaled(LAST, mt - 1);
#pragma unroll
        for (int i = 0; i < ST && t0 + i < NT; ++i) held[i] = part[i];
      }
      if (mt == MT - 1) add_scaled(LAST, mt);
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int t = 0; t < NT; ++t)
          acc[t][mtc] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A[t][j], v[j], acc[t][mtc], 0, 0, 0);
    }
  };
  auto landed = [&]() BK_INLINE {  // after a wait: what was waited for is read from here on
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };

  // between a wave's units: where the next one begins another window, every wave is done with this one
  [[maybe_unused]] auto next_window = [&]() BK_INLINE {
    ++done;
    if (windows && done % window == 0 && done < units_most) {
      asm volatile("s_barrier" ::: "memory");
      copy_window(done / window);
      g_first += GP;
      asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
    }
  };

  if constexpr (AHEAD) {
    // A piece is read back while the one before it is multiplied (few row tiles: N = 4096, K = 14336, M = 64
    // 19.7 -> 17.9 us; with larger blocks the second set of registers costs more than it gives).
    h8 xv[2][4];
    if (nu > 0) {
      __builtin_amdgcn_s_waitcnt(waitcnt_vm(4 * (XS - 1)));
      landed();
      read_codes(0, cw[0]), read_codes(1, cw[1]);
      read_x(0, xv[0]);
      read_params(2 * wave);
    }
    for (int U = wave; U < units; U += BK_WAVES) {
      const bool more = U + BK_WAVES < units;
      bk_for([&](auto pc) BK_INLINE {
        constexpr int p = decltype(pc)::value, ch = p / MT, mt = p % MT;
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): this piece is in registers and its place free
        landed();
        request_next(pc, U, more);
        scale_t scale[NT];
        zero_t zword[NT];
        const int group = g;
        if (mt == 0) {
#pragma unroll
          for (int t = 0; t < NT; ++t) {
            scale[t] = sc[t];
            if (FMT == 1) zword[t] = zw[t];
          }
        }
        // requests younger than the next piece: the ring's others and, early in a unit, the next unit's codes
        if (p + 1 < NP || more) {
          constexpr int left = NP - 2 - p < 0 ? 0 : NP - 2 - p < XS - 1 ? NP - 2 - p : XS - 1;
          if (more) __builtin_amdgcn_s_waitcnt(waitcnt_vm(4 * (XS - 1) + (p < XS - 1 ? CL : 0)));
          else __builtin_amdgcn_s_waitcnt(waitcnt_vm(4 * left));
          landed();
          if (MT > 1 && p == NP - 1) read_codes(0, cw[0]), read_codes(1, cw[1]);
          read_x(slot, xv[(p + 1) & 1]);
          if (p == MT - 1) read_params(2 * U + 1);
          if (p == NP - 1) {
            if constexpr (GM == 2) next_window();
            read_params(2 * (U + BK_WAVES));
          }
        }
        __builtin_amdgcn_sched_barrier(0);
        if (mt == 0) expand(cw[ch], scale, zword, group, U * BK_UNIT + ch * 128 + 32 * b);
        multiply(std::integral_constant<int, mt>{}, 2 * U + ch, xv[p & 1]);
        if (MT == 1 && p == NP - 1 && more) read_codes(0, cw[0]), read_codes(1, cw[1]);
        __builtin_amdgcn_sched_barrier(0);
      }, std::make_integer_sequence<int, NP>{});
    }
    if constexpr (GM == 2) next_window();  // (a wave without a unit in the last window meets the others there)
  } else {
    for (int U = wave; U < units; U += BK_WAVES) {
      const bool more = U + BK_WAVES < units;
      bk_for([&](auto pc) BK_INLINE {
        constexpr int p = decltype(pc)::value, ch = p / MT, mt = p % MT;
        // requests younger than the ones needed: the ring's other pieces, and next unit's codes
        constexpr int R = XS - 1, left = NP - 1 - p < R ? NP - 1 - p : R;
        if (more) __builtin_amdgcn_s_waitcnt(waitcnt_vm(4 * R + (p > PC && p < PC + XS ? CL : 0)));
        else __builtin_amdgcn_s_waitcnt(waitcnt_vm(4 * left));
        landed();
        if (PC && mt == 0) read_codes(ch, cw[0]);
        if (!PC && p == 0) read_codes(0, cw[0]), read_codes(1, cw[PC ? 0 : 1]);
        h8 xv[4];
        read_x(slot, xv);
        if (mt == 0) read_params(2 * U + ch);
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the places are free
        landed();
        request_next(pc, U, more);
        __builtin_amdgcn_sched_barrier(0);
        if (mt == 0) expand(cw[PC ? 0 : ch], sc, zw, g, U * BK_UNIT + ch * 128 + 32 * b);
        multiply(std::integral_constant<int, mt>{}, 2 * U + ch, xv);
        __builtin_amdgcn_sched_barrier(0);
      }, std::make_integer_sequence<int, NP>{});
    }
  }

  // ---- the waves' sums, added in wave order; PH row tiles at a time, as LDS holds ----
  constexpr int PH = (BK_WAVES * WB) / (BK_WAVES * NT * 1024) < MT ? (BK_WAVES * WB) / (BK_WAVES * NT * 1024) : MT;
  f4* const red = (f4*)bk_lds;  // [wave][t][PH][64]
#pragma unroll
  for (int mb = 0; mb < MT; mb += PH) {
    __syncthreads();
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int i = 0; i < PH; ++i)
        if (mb + i < MT) red[((wave * NT + t) * PH + i) * 64 + lane] = acc[t][mb + i];
    __syncthreads();
    // a thread makes 8 consecutive outputs of one activation row: 2 NT of them are the row's 16 NT
    for (int e = (int)threadIdx.x; e < PH * 16 * 2 * NT; e += BK_THREADS) {
      const int seg = e % (2 * NT), row = e / (2 * NT), i = row >> 4, rr = row & 15, t = seg >> 1;
      const int m = m0 + 16 * (mb + i) + rr, n = n0 + 8 * seg;
      if (mb + i >= MT || m >= M || n >= N) continue;
      const int at = (t * PH + i) * 64 + 32 * (seg & 1) + rr;
      f4 s0 = red[at], s1 = red[at + 16];
#pragma unroll
      for (int w = 1; w < BK_WAVES; ++w) {
        s0 += red[w * NT * PH * 64 + at];
        s1 += red[w * NT * PH * 64 + at + 16];
      }
      const h8 hv = h8{(_Float16)s0[0], (_Float16)s0[1], (_Float16)s0[2], (_Float16)s0[3],
                       (_Float16)s1[0], (_Float16)s1[1], (_Float16)s1[2], (_Float16)s1[3]};
      w4_half* const dst = c + (size_t)m * N + n;
      if (RAG && (N & 7)) {
        const int left = N - n;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const _Float16 h = hv[j];  // (a bit cast of a vector's element takes the first)
          if (j < left) dst[j] = __builtin_bit_cast(uint16_t, h);
        }
      } else {
        *(h8*)dst = hv;
      }
    }
  }
}

bool bk_ragged(const WView& v) { return v.K % 32 || v.N % 16; }

// Bytes of LDS of a workgroup with NT tiles of W, of whose rows it has the parameters of G groups.
int bk_lds_bytes(const WView& v, int NT, int G) {
  const long long p = 16LL * NT * G * (v.mx ? 1 : 2), z = v.mx || v.symmetric ? 0 : 64LL * NT * words(G);
  const int slack = !v.mx && (v.gs % 32 || bk_ragged(v)) ? 16 : 0;  // GM: the last dword of a run may lie behind the parameters
  const long long bytes = BK_WAVES * bk_wave_bytes(NT, BK_XS) + ((p + 1023) & ~1023LL) + ((z + 1023) & ~1023LL) + slack;
  return bytes > (1 << 20) ? 1 << 20 : (int)bytes;
}
int bk_lds_bytes(const WView& v, int NT) { return bk_lds_bytes(v, NT, v.mx ? v.B : v.G); }
constexpr int BK_MAX_LDS = 160 * 1024;

// Units of a wave whose parameters LDS holds at a time: all (BK_WHOLE), or as many as fit, where a unit is whole groups
// and rows are whole dwords; 0: not even one's.
constexpr int BK_WHOLE = 1 << 20;
int bk_window(const WView& v, int NT) {
  if (bk_lds_bytes(v, NT) <= BK_MAX_LDS) return BK_WHOLE;
  if (v.mx || v.gs >= 32 || 32 % v.gs || v.G % 2) return 0;
  int w = ((v.K + BK_UNIT - 1) / BK_UNIT + BK_WAVES - 1) / BK_WAVES;
  while (w > 0 && bk_lds_bytes(v, NT, w * (BK_WAVES * BK_UNIT / v.gs)) > BK_MAX_LDS) --w;
  return w;
}

template <int FMT, int NT, int MT, bool LATE, int GM, bool RAG>
hipError_t block_go_as(const WView& v, const w4_half* x, w4_half* c, int M, hipStream_t s, w4_half* w_out) {
  constexpr int XS = BK_XS;
  constexpr bool AHEAD = NT <= 2;
  const int window = GM == 2 ? bk_window(v, NT) : BK_WHOLE;
  if (window < 1) return hipErrorInvalidValue;
  const int lds_bytes = window == BK_WHOLE ? bk_lds_bytes(v, NT) : bk_lds_bytes(v, NT, window * (BK_WAVES * BK_UNIT / v.gs));
  static std::atomic<bool> granted[64] = {};  // more than 64 KB of LDS has to be granted per device, once
  int dev = 0;
  if (hipError_t e = hipGetDevice(&dev); e != hipSuccess) return e;
  if (dev < 0 || dev >= 64 || !granted[dev]) {
    const hipError_t e = hipFuncSetAttribute((const void*)mfma_block_kernel<FMT, NT, MT, XS, AHEAD, LATE, GM, RAG>,
                                             hipFuncAttributeMaxDynamicSharedMemorySize, BK_MAX_LDS);
    if (e != hipSuccess) return e;
    if (dev >= 0 && dev < 64) granted[dev] = true;
  }
  const uint32_t mg = (M + 16 * MT - 1) / (16 * MT), ng8 = ((uint32_t)v.N + 128 * NT - 1) / (128 * NT);
  const dim3 grid(8 * mg, ng8 < BK_GRID_Y ? ng8 : BK_GRID_Y, (ng8 + BK_GRID_Y - 1) / BK_GRID_Y);
  const uint32_t mul = v.mx ? 0u : (uint32_t)(((1ULL << 31) + v.gs / 8 - 1) / (v.gs / 8));
  mfma_block_kernel<FMT, NT, MT, XS, AHEAD, LATE, GM, RAG><<<grid, BK_THREADS, lds_bytes, s>>>(
      v.q, v.scales, v.zeros, x, c, v.N, v.K, M, v.mx ? v.B : v.G, v.gs, mul, window, w_out);
  return hipGetLastError();
}

// Forms that are compiled for blocks of NT x MT.  Rows of words that are only 4-byte aligned take four times the load
// instructions, small groups take LDS for their parameters: neither has blocks of more than two tiles of W.
constexpr bool bk_has(int fmt, int NT, int gm, bool rag) {
  return fmt == 2 || gm == 0 || NT <= 2 || (gm == 1 && !rag);
}

template <int FMT, int NT, int MT>
hipError_t block_go(const WView& v, const w4_half* x, w4_half* c, int M, hipStream_t s, w4_half* w_out) {
  const bool rag = bk_ragged(v);
  if constexpr (FMT == 2) {
    return rag ? block_go_as<2, NT, MT, false, 0, true>(v, x, c, M, s, w_out) : block_go_as<2, NT, MT, false, 0, false>(v, x, c, M, s, w_out);
  } else {
    const int gm = v.gs < 32 ? 2 : rag || v.gs % 32 ? 1 : 0;
    if (gm == 0)
      return v.gs % 128 == 0 ? block_go_as<FMT, NT, MT, true, 0, false>(v, x, c, M, s, w_out)
                             : block_go_as<FMT, NT, MT, false, 0, false>(v, x, c, M, s, w_out);
    if constexpr (bk_has(FMT, NT, 1, false))
      if (gm == 1 && !rag) return block_go_as<FMT, NT, MT, false, 1, false>(v, x, c, M, s, w_out);
    if constexpr (bk_has(FMT, NT, 1, true))
      if (gm == 1 && rag) return block_go_as<FMT, NT, MT, false, 1, true>(v, x, c, M, s, w_out);
    if constexpr (bk_has(FMT, NT, 2, false))
      if (gm == 2 && !rag) return block_go_as<FMT, NT, MT, false, 2, false>(v, x, c, M, s, w_out);
    if constexpr (bk_has(FMT, NT, 2, true))
      if (gm == 2 && rag) return block_go_as<FMT, NT, MT, false, 2, true>(v, x, c, M, s, w_out);
    return hipErrorInvalidValue;
  }
}

// Blocks and what a wave needs for 128 k of one, in units of 10 ns, W4 and MXFP4 (N = 4096, K = 14336 with
// as many rows as make one round of workgroups, and N = 5120, K = 13824; a call takes 3.5 us more).  Groups of whole
// chunks cost 0.97 to 1.03 of it.
// The time of a call is start + rounds of workgroups x (round + per_n x units of the first wave + store), per_n for symmetric
// W4, W4 with zero-points and MXFP4, store where N is no multiple of 8 and halves leave one by one.  any: shapes that are not
// whole tiles, chunks and groups (MXFP4: as RAG), fitted to 8000 of 5 to 4000 rows, K = 256 to 14336, to within 8 to 10 %
// (r.m.s.); whole: the others.
struct BkTime {
  int start, round, per_n[3], store;
};
struct BkShape {
  int nt, mt, cost_w4, cost_mx;
  BkTime whole, any;
};
constexpr BkShape BK_SHAPES[] = {
    {1, 1, 50, 45, {170, 130, {118, 133, 99}, 0}, {149, 134, {104, 114, 95}, 20}},
    {2, 1, 83, 56, {140, 150, {188, 211, 139}, 0}, {118, 184, {162, 182, 139}, 23}},
    {2, 2, 106, 89, {85, 210, {228, 247, 200}, 0}, {114, 199, {197, 217, 192}, 37}},
    {4, 1, 136, 80, {110, 150, {334, 382, 223}, 0}, {134, 192, {319, 335, 236}, 24}},
    {2, 4, 171, 155, {5, 300, {320, 335, 314}, 0}, {79, 254, {283, 302, 373}, 50}},
    {4, 2, 175, 125, {70, 240, {390, 443, 303}, 0}, {78, 296, {362, 415, 306}, 33}},
    {3, 4, 195, 173, {-20, 370, {397, 426, 378}, 0}, {-18, 412, {416, 401, 395}, 100}},
    {4, 4, 260, 215, {-45, 370, {505, 543, 458}, 0}, {-37, 448, {504, 485, 491}, 110}},
    {4, 5, 290, 250, {-100, 450, {570, 617, 550}, 0}, {-75, 516, {543, 529, 560}, 90}},
    {4, 6, 330, 290, {-110, 490, {624, 668, 634}, 0}, {-82, 586, {605, 626, 621}, 110}}};
constexpr int BK_COUNT = sizeof BK_SHAPES / sizeof BK_SHAPES[0];

long long bk_rounds(const WView& v, int M, const BkShape& s, int cus) {
  const long long ng = (v.N + 16 * s.nt - 1) / (16 * s.nt), mg = (M + 16 * s.mt - 1) / (16 * s.mt);
  return ((ng + 7) / 8 * mg + cus / 8 - 1) / (cus / 8);
}

// Small groups take 0.035 us for every KB of a block's parameters, which are copied first (N = 11008, K = 4096, gs = 8, M = 16,
// 32 x 16 blocks 15.7 us, the decode kernel 14.0), and 4.5 us for another window of them; codes by the dword and rows past N
// 1.23 of W4's units.  From three rounds on a call takes 1.08 of the sum (M = 789, N = 2896, K = 11680, gs = 40, twelve rounds
// of 32 x 64: 137 us, tiles 97).
int bk_time(const WView& v, int M, const BkShape& s, int cus, bool whole) {
  const BkTime& b = whole ? s.whole : s.any;
  const int n = ((v.K + BK_UNIT - 1) / BK_UNIT + BK_WAVES - 1) / BK_WAVES;
  const long long per = b.per_n[v.mx ? 2 : v.symmetric ? 0 : 1] * (!v.mx && bk_ragged(v) ? 123 : 100) / 100;
  const long long copy = v.mx || v.gs >= 32 ? 0 : 16LL * s.nt * (2 * v.G + (v.symmetric ? 0 : 4 * words(v.G))) * 7 / 2048;
  const int window = copy ? bk_window(v, s.nt) : BK_WHOLE, more = window > 0 && window < n ? (n - 1) / window : 0;
  const long long rounds = bk_rounds(v, M, s, cus);
  const long long sum = b.start + rounds * (b.round + copy + per * n + 450 * more + (v.N % 8 ? b.store : 0));
  const long long t = rounds > 2 && !whole ? sum * 108 / 100 : sum;
  return t > 1 << 30 ? 1 << 30 : (int)t;
}

// Few rows (M < 17) and at most one tile of W a compute unit, K in whole chunks: the longest K that stays with the long-K
// kernel, which fetches only the quads of x that exist and has no parameters to wait for.  [symmetric W4, with
// zero-points, MXFP4][M up to 4, 8, 12, 16][tiles for half of the compute units, or more].  M = 3: N = 128, K = 5120 5.5 us
// against 4.5, N = 4096, K = 6144 7.3 against 6.4; M = 7: N = 1024, K = 4224 6.0 against 5.2; M = 11: N = 128, K = 4352 5.0
// against 4.7.  At K = 14336 blocks are 1.05 (M = 4) to 1.3 times (M = 16) as fast.
constexpr int BK_LONGEST[3][4][2] = {{{1 << 30, 10240}, {8192, 6144}, {6144, 0}, {5120, 0}},
                                     {{6144, 5120}, {6143, 5120}, {4608, 0}, {4096, 0}},
                                     {{9216, 7168}, {6144, 5120}, {5120, 0}, {4096, 0}}};

// Whether blocks of shape s in `rounds` rounds of workgroups are ahead of the kernel that has the call otherwise.
// That kernel is told apart by the same arithmetic as in the dispatcher and the kernels' own rules. The lines come
// from 10800 shapes of 3 to 3000 rows, both kernels timed in turn.  Few tiles or a short K leave a block its start
// and the sum of eight waves.
bool block_ahead(const WView& v, int M, const BkShape& s, long long rounds, bool dma, int cus) {
  const int tiles = v.N / 16, area = s.nt * s.mt, units = (v.K + BK_UNIT - 1) / BK_UNIT, K = v.K;
  const bool whole = K % 128 == 0, sym = !v.mx && v.symmetric;
  if (M < 17) {
    // up to 8 rows in blocks of 64: N = 11008, K = 13824, M = 4 37.6 us against 32.5 (M = 13 36.3 against 49.6)
    if (s.mt > 1 && M < 9) return false;
    // MXFP4 in no whole chunks: behind on a few tiles of a short row only (N = 128, K = 4128, M = 5 4.7 us against 4.3)
    if (!whole) return !v.mx || 8 * tiles >= cus || K >= (M < 9 ? 6144 : 3072);
    // four tiles of symmetric W4, whose expansion bounds them, for 3 or 4 rows, where the other kernel has up to three
    // rounds: N = 11008, K = 6144 15.5 against 14.1 (N = 13824, K = 5120 14.5 against 17.0)
    if (tiles > cus) return s.nt < 4 || M > 4 || !sym || tiles > 3 * cus;
    if (K < 4096) return false;  // M = 11: N = 128, K = 2304 4.4 against 4.0; M = 14: N = 1024, K = 3072 5.1 against 4.6
    // W4 with whole-chunk groups, whose scales the resident kernel has in registers: N = K = 4096, gs = 128, M = 12 / 16
    // 6.0 / 6.2 us against 5.6 / 6.0 (gs = 64 5.9 / 6.1 against 5.9 / 6.3)
    if (K == 4096 && !v.mx && v.gs % 128 == 0 && 2 * tiles > cus) return false;
    return K > BK_LONGEST[v.mx ? 2 : sym ? 0 : 1][(M - 1) / 4][2 * tiles >= cus];
  }
  if (whole && M <= 64 && tiles <= cus && K > 1024 && K != 2048 && K != 4096) {
    // the long-K kernel again: N = 2576, K = 1664, gs = 96, M = 43 7.9 us in two rounds against 5.7; more than one tile
    // a block where it has one a compute unit: N = 3952, K = 1920, M = 17 5.7 against 4.9, K = 2688 6.4 against 5.7
    if (rounds > 1) return false;
    return 2 * tiles <= cus || area < 2 || K >= (area == 2 && !v.mx ? 3072 : 2048);
  }
  if (M >= 65 && dma && (long long)((v.N + 255) / 256) * ((M + 127) / 128) >= 8) {
    // Direct-to-LDS tiles.  A block's size is bounded by the units of K it has to work through: K = 1152, N = 8192, M = 72
    // 10.5 us against 8.5 (64 x 64), N = 4096, M = 89 7.4 against 8.7 (32 x 64); nine units are two for one wave and
    // one for the others: K = 2304, N = 6144, M = 146 12.4 against 9.9.
    // N = 288, K = 11904, M = 2857 84.6 against 57.4; N = 544, K = 4608 (18 units), M = 1256 21.1 against 18.5
    if (M > 1536 || (M > 1024 && v.N >= 256 && 32 * ((units + 7) / 8) > 5 * units)) return false;
    // gs = 32 with zero-points has two smallest tiles of its own there, which are behind from four units on (M = 95, N = 14416,
    // K = 3072 16.3 against 25.6); shorter K: M = 68, N = 5712, K = 384 7.1 against 6.0, N = 4784, M = 118 7.1 and 6.1, K = 640,
    // N = 6464, M = 66 8.0 and 7.4 (2700 calls: blocks of up to 8 tiles of 16 x 16 at two units and 12 at three are ahead)
    if (!v.mx && !sym && v.gs == 32) {
      constexpr int largest32[5] = {0, 2, 8, 12, 20};
      return units > 4 || area <= largest32[units];
    }
    constexpr int largest[14] = {0, 2, 2, 4, 8, 8, 12, 12, 24, 12, 20, 20, 20, 20};
    return units > 13 || area <= largest[units];
  }
  // What those tiles do not take; several rounds pay there as well (K = 9760, N = 3072, M = 448: 105 -> 69 us in two).
  if (M >= 96 && K % 64 == 0) {
    // Register-staged tiles of 256 x 128, which are ahead where they fill their own rounds.  In rounds of 64 x 96 blocks:
    // N = 8192, K = 1088, M = 984 69 us in four against 38; K = 5120, gs = 96, M = 895 121 in five against 104 (256
    // tiles), N = 13824, M = 667 132 in six against 182 (324); N = 5120, K = 13824, M = 1140 211 in four against 270.
    const long long others = (long long)((M + 255) / 256) * ((v.N + 127) / 128), other_rounds = (others + cus - 1) / cus;
    if (8 * others < cus) return true;
    const long long load = rounds * (v.mx ? s.cost_mx : s.cost_w4), r = (load + 329) / 330;
    constexpr int shortest[5] = {0, 0, 512, 1024, 2304};
    return K >= (r < 5 ? shortest[r] : 3072) && (r < 4 || load < (K < 6144 ? 1320 : 1980) * other_rounds);
  }
  // The stream kernel.  N = 8736, K = 512, M = 28 6.0 us in 64 x 32 blocks against 4.6; N = 1120, K = 256, M = 45 in
  // 64 x 16 4.5 against 4.7; N = 592, K = 9248, M = 2834 144 in three rounds against 119
  if (rounds == 1) return area <= (K <= 512 ? 4 : K < 768 ? 12 : 24);
  return K >= (rounds == 2 ? 768 : 1024) && (M <= 1536 || rounds == 2);
}

// The block that covers the call in the least time (rounds of workgroups x cost of one), as an index into
// BK_SHAPES; -1: none, or another kernel is ahead.
int block_plan(const WView& v, int M) {
  if (M < 3 || M > 8192 || (M < 9 && v.K <= 4096) || (M < 17 && v.K <= 2048)) return -1;
  if (v.K % 32 || v.N % 16 || (!v.mx && v.gs % 32)) return -1;
  if (v.K >= 1 << 24 || !any_group_fits(v)) return -1;  // offsets inside a block have 32 bits
  const int cus = device_cus();
  if (cus < 8) return -1;
  // Few rows: one 16-row tile of W a workgroup (N = K = 4096, M = 8 5.2 against 5.0 us; K = 2048, M = 16 4.2 against
  // 3.9), wider matrices at long K only (N = 11008, K = 4096, M = 16 9.4 against 7.7 us).  (Ruled out first: calls this
  // short see host time.)
  if (M < 17 && v.K <= 4096 && v.N > 16 * cus) return -1;
  // The direct-to-LDS tile kernel's operands: one round of workgroups only (K = 8192, N = 8192, M = 256: two take 50 us
  // against its 48).
  const bool dma = v.K % 128 == 0 && (v.mx || v.gs == 32 || v.gs == 64 || v.gs % 128 == 0);
  int best = -1;
  long long least = 0, best_rounds = 0;
  for (int i = 0; i < BK_COUNT; ++i) {
    const BkShape& s = BK_SHAPES[i];
    if (bk_lds_bytes(v, s.nt) > BK_MAX_LDS) continue;
    const long long rounds = bk_rounds(v, M, s, cus);
    if (rounds > (dma || M < 17 ? 1 : 8)) continue;
    const long long cost = rounds * (v.mx ? s.cost_mx : s.cost_w4);
    if (best < 0 || cost < least) best = i, least = cost, best_rounds = rounds;
  }
  if (best < 0 || !block_ahead(v, M, BK_SHAPES[best], best_rounds, dma, cus)) return -1;
  if (!dma) return best;
  // One round at K of one or two units a wave and many rows: N = 4096, K = 1024, M = 192 7.8 against 6.9 us,
  // K = 2048, M = 333 12.1 against 10.9.
  if ((v.K < 2048 && M > 128) || (v.K < 4096 && M > 256)) return -1;
  // Up to 32 rows of wide matrices at the resident kernel's own K: N = 11008, M = 32 12.4 against 10.4 us; W4 at the
  // shorter of the two always: N = 2048, M = 32 5.1 against 4.9.
  if (M <= 32 && (v.K == 2048 || v.K == 4096) && BK_SHAPES[best].nt == 4) return -1;
  if (M <= 32 && v.K == 2048 && !v.mx) return -1;
  return best;
}

template <int FMT>
hipError_t block_fmt(int shape, const WView& v, const w4_half* x, w4_half* c, int M, hipStream_t s, w4_half* w_out) {
  switch (shape) {
    case 0: return block_go<FMT, 1, 1>(v, x, c, M, s, w_out);
    case 1: return block_go<FMT, 2, 1>(v, x, c, M, s, w_out);
    case 2: return block_go<FMT, 2, 2>(v, x, c, M, s, w_out);
    case 3: return block_go<FMT, 4, 1>(v, x, c, M, s, w_out);
    case 4: return block_go<FMT, 2, 4>(v, x, c, M, s, w_out);
    case 5: return block_go<FMT, 4, 2>(v, x, c, M, s, w_out);
    case 6: return block_go<FMT, 3, 4>(v, x, c, M, s, w_out);
    case 7: return block_go<FMT, 4, 4>(v, x, c, M, s, w_out);
    case 8: return block_go<FMT, 4, 5>(v, x, c, M, s, w_out);
    default: return block_go<FMT, 4, 6>(v, x, c, M, s, w_out);
  }
}

}  // namespace

int block_plan_time(const WView& v, int M, int* time) {
  const int i = block_plan(v, M);
  if (i >= 0) *time = bk_time(v, M, BK_SHAPES[i], device_cus(), true);
  return i;
}

int block_any_time(const WView& v, int M, int cus, int* time) {
  // (more rows of x than L2 holds, which every block of W reads again, are the tiles': N = 276, K = 11104, M = 3020 143 us
  // in 32 x 64 blocks)
  if (v.K % 8 || v.K < 32 || v.K >= 1 << 24 || M > 1536 || !any_group_fits(v)) return -1;
  const int gm = v.mx ? 0 : v.gs < 32 ? 2 : 1;
  int best = -1;
  for (int i = 0; i < BK_COUNT; ++i) {
    const BkShape& s = BK_SHAPES[i];
    if (!bk_has(v.mx ? 2 : 0, s.nt, gm, bk_ragged(v)) || bk_window(v, s.nt) < 1) continue;
    const int t = bk_time(v, M, s, cus, false);
    if (best < 0 || t < *time) best = i, *time = t;
  }
  return best;
}

int block_shape(const WView& v, int M) {
  const AnyPlan any = any_plan(v, M);
  const int i = any.kind == 1 ? any.shape : any.kind == 3 ? -1 : block_plan(v, M);
  return i < 0 ? 0 : 10 * BK_SHAPES[i].nt + BK_SHAPES[i].mt;
}

bool try_block(const WView& v, const w4_half* x, w4_half* c, int M, hipStream_t s, w4_half* w_out, int shape, hipError_t* err) {
  if (((uintptr_t)v.q | (uintptr_t)v.scales | (uintptr_t)v.zeros | (uintptr_t)x | (uintptr_t)c | (uintptr_t)w_out) & 15)
    return false;
  if (shape < 0) shape = block_plan(v, M);
  if (shape < 0) return false;
  if (v.mx) *err = block_fmt<2>(shape, v, x, c, M, s, w_out);
  else if (v.symmetric) *err = block_fmt<0>(shape, v, x, c, M, s, w_out);
  else *err = block_fmt<1>(shape, v, x, c, M, s, w_out);
  return true;
}

}  // namespace w4k
