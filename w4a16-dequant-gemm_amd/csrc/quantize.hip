// Device-side quantizers: the host quantizers of the packed formats as gfx950
// kernels, producing the same bytes.
//
//   rows of W4 codes (weights and KV-cache rows) ... pack.hpp:64-130, kvcache.hpp:60-108
//   rows of E4M3 bytes (FP8 KV cache) ............... kvfp8.hpp:70-128
//   rows of MXFP4 codes ............................. mx.hpp:71-119
//
// Bit identity with the host comes from doing the same IEEE operations in the
// same order: min/max and the step in FP64, the step rounded FP64 -> FP32 ->
// FP16 in two hardware conversions (both round to nearest even, FP16
// subnormals kept), every element divided in FP64 by the stored scale, and
// round-half-away-from-zero done on the exact fraction.  The MXFP4 block
// exponent is the smallest e with amax <= 6 * 2^e, which is what the host's
// ceil(log2(amax / 6)) followed by its upward fix-up loop evaluates to; here
// it is read off the exponent field and settled by one exact comparison.
//
// The kernels are memory-bound streams: one thread per packed word (8 elements
// in, 4 or 8 bytes out), group extrema combined through LDS.  Conditions the
// host reports by throwing (non-finite input, scale outside the FP16 / E8M0
// range) are OR-ed into a caller-provided status word: bit 0 non-finite input,
// bit 1 scale out of range.  Outputs are unspecified when it ends non-zero.
#include <float.h>

#include <mutex>

#include "dq.cuh"
#include "kernels.h"

namespace w4k {
namespace {

constexpr int QT = 256;  // threads per workgroup

// The caller's status word, which a call first clears and then ORs what it found into.  A launch of
// its own for the clearing was 2.5 us of a call of 7 (8 x 4096 x 128 keys and values) and of 6 (one row);
// so the word is cleared once by whoever comes first, the first workgroup or a lane that has something to
// report (which is rare): the first to leave the call's ticket in qz_claimed clears and then says so in
// qz_cleared, and a reporting lane waits for that before it ORs.  It waits for a wave that is running and a few
// instructions from the end of the wait, never for a workgroup that has yet to be placed: the XCD of the
// first workgroup may be full of another stream's work for any time.
// A slot belongs to one stream, whose calls run one after the other with ascending tickets (StatusCall): no
// other call can take the slot over between two arrivals of a call, which would clear the word again.
// Tickets only ever replace lower ones, so that what may be left of a stream destroyed with work in
// flight takes nothing from a stream that has its address.
// Stores and loads at agent scope and a wait for the store in between are the order that is needed, as in
// the flash kernels' merge; a release fence would write a whole L2 back.
// ticket: the call's number in its slot x QZ_SLOTS + the slot; 0: an earlier launch has cleared the word.
// (One word, so that all arguments of a kernel arrive in registers.)
constexpr int QZ_SLOTS = 64;
typedef unsigned long long qz_ticket;
__device__ qz_ticket qz_claimed[QZ_SLOTS], qz_cleared[QZ_SLOTS];
struct Status {
  int* word;
  qz_ticket ticket;
};

__device__ __forceinline__ void clear_once(const Status& st) {
  const uint32_t slot = (uint32_t)st.ticket % QZ_SLOTS;
  if (__hip_atomic_fetch_max(&qz_claimed[slot], st.ticket, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < st.ticket) {
    __hip_atomic_store(st.word, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __hip_atomic_fetch_max(&qz_cleared[slot], st.ticket, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

__device__ __forceinline__ void begin_status(const Status& st) {
  if (st.ticket && (blockIdx.x | blockIdx.y | threadIdx.x) == 0) clear_once(st);
}

// Only what is not there yet takes an atomic: with input full of NaN every lane reports, and a claim and an
// OR each take 270 us for 8 x 4096 x 128 keys and values (as an exchange, which the compiler does not
// merge over a wave, 11.9 ms); two loads take 93.
__device__ __forceinline__ void report(const Status& st, int bits) {
  if (st.ticket) {
    qz_ticket* const cleared = &qz_cleared[(uint32_t)st.ticket % QZ_SLOTS];
    if (__hip_atomic_load(cleared, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < st.ticket) {
      clear_once(st);
      for (int n = 0; n < 65536; ++n) {
        if (__hip_atomic_load(cleared, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) >= st.ticket) break;
        __builtin_amdgcn_s_sleep(4);
      }
    }
  }
  if ((__hip_atomic_load(st.word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & bits) != bits) atomicOr(st.word, bits);
}

__global__ void fill_words_kernel(uint32_t* p, long long n, uint32_t value) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = value;
}

enum { QM_SYM = 0, QM_ASYM = 1, QM_F8 = 2 };

// Up to two independent jobs of the same shape in one launch (the K and the V
// side of a cache): blockIdx.y picks the side.
template <typename T>
struct Sides {
  const T* src[2];
  uint32_t* q32[2];
  uint8_t* q8[2];
  uint16_t* scales[2];
  uint32_t* zeros[2];
};

// lround() for |v| far below 2^52: the fraction v - trunc(v) is exact.
__device__ __forceinline__ long round_half_away(double v) {
  double t = trunc(v);
  const double frac = fabs(v - t);
  t = fmin(fmax(t, -1.0e12), 1.0e12);
  long r = (long)t;
  if (frac >= 0.5) r += v < 0.0 ? -1 : 1;
  return r;
}

__device__ __forceinline__ int clamp_code(long v) { return (int)(v < 0 ? 0 : (v > 15 ? 15 : v)); }

__device__ __forceinline__ bool finite(double x) { return fabs(x) <= DBL_MAX; }

// kvfp8.hpp:48-53 (the encoder of quantize_cache_f8): round to nearest even on
// the E4M3 grid, saturate at 448, NaN -> 0x7F.
__device__ __forceinline__ uint32_t encode_e4m3(float x) {
  const uint32_t bits = __builtin_bit_cast(uint32_t, x);
  const uint32_t sign = (bits >> 24) & 0x80u;
  const float a = fabsf(x);
  if (a != a) return sign | 0x7Fu;
  if (a >= 448.0f) return sign | 0x7Eu;
  int ex = (int)((bits >> 23) & 0xFFu) - 127;
  if (ex < -6) ex = -6;
  // a * 2^(3 - ex) is exact; one rint is the rounding (0..16 steps)
  const int steps = (int)rintf(a * __builtin_bit_cast(float, (uint32_t)(130 - ex) << 23));
  const int code = (ex == -6 && steps < 8) ? steps : (ex + 7) * 8 + (steps - 8);
  return sign | (uint32_t)(code > 0x7E ? 0x7E : code);
}

// Four E4M3 bytes of FP32 values that are not NaN (the hardware conversion rounds to nearest even,
// subnormals included; past 448 it would give NaN, so the magnitude is capped first).  `from`
// gives the signs.
__device__ __forceinline__ uint32_t pack_e4m3(const float* mag, const float* from) {
  float x[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) x[i] = copysignf(fminf(mag[i], 448.0f), from[i]);
  const int lo = __builtin_amdgcn_cvt_pk_fp8_f32(x[0], x[1], 0, false);
  return (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(x[2], x[3], lo, true);
}

// |v / s| for FP16-representable v and s > 0, near enough for E4M3 without the division: x = |v| * rs
// with rs = 1 / s to within 2^-22, then one correction by the residual |v| - x s, which is
// exact (a multiple of ulp(x) ulp(s) that is 2^-21 of |v|: under 24 bits).  The exact quotient has
// an 11-bit numerator and denominator: it is either on a midpoint of the E4M3 grid, which has 5
// bits and which the correction then returns exactly, or at least 2^-16 (relative) away from
// every midpoint, so that x rounds as it does.  (The host rounds the FP64 quotient to FP32 first,
// which for the same reason never moves it onto or across a midpoint.)
__device__ __forceinline__ float quotient_magnitude(float v, float s, float rs) {
  const float a = fabsf(v), x = a * rs;
  return fmaf(fmaf(-x, s, a), rs, x);
}

__device__ __forceinline__ int pow2_at_least(int n) {
  int p = 1;
  while (p < n) p <<= 1;
  return p;
}

// One workgroup quantizes QT / tpg consecutive (row, group) pairs, tpg =
// min(gs / 8, QT) threads each; a thread owns whole packed words.  T is the
// source element type (double or _Float16).
template <typename T, int MODE>
__global__ __launch_bounds__(QT) void quantize_rows_kernel(
    const Sides<T> sd, long long rows, int K, int gs, int G, const Status status) {
  begin_status(status);
  const T* __restrict__ src = sd.src[blockIdx.y];
  uint32_t* __restrict__ q32 = sd.q32[blockIdx.y];
  uint8_t* __restrict__ q8 = sd.q8[blockIdx.y];
  uint16_t* __restrict__ scales = sd.scales[blockIdx.y];
  uint32_t* __restrict__ zeros = sd.zeros[blockIdx.y];
  __shared__ double s_lo[QT], s_hi[QT];
  __shared__ float s_scale[QT];
  __shared__ int s_zero[QT];

  const int wpg = gs >> 3;
  const int tpg = wpg < QT ? wpg : QT;
  const int gpb = QT / tpg;
  const int t = threadIdx.x;
  const int lg = t / tpg, li = t - lg * tpg;
  const long long gid = (long long)blockIdx.x * gpb + lg;
  const bool live = lg < gpb && gid < rows * G;
  long long row = 0;
  int g = 0;
  if (live) {
    row = gid / G;
    g = (int)(gid - row * G);
  }
  const int k0 = g * gs;
  const int len = live ? (gs < K - k0 ? gs : K - k0) : 0;
  const int nw = (len + 7) >> 3;
  const T* base = src + row * (long long)K + k0;

  // extrema of this thread's words; the first word stays in registers
  double lo = INFINITY, hi = -INFINITY;
  double first[8];
  bool bad = false;
#pragma unroll
  for (int j = 0; j < 8; ++j) first[j] = 0.0;
  for (int wi = li; wi < nw; wi += tpg) {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int e = wi * 8 + j;
      if (e < len) {
        const double x = (double)base[e];
        bad |= !finite(x);
        lo = fmin(lo, x);
        hi = fmax(hi, x);
        if (wi == li) first[j] = x;
      }
    }
  }
  if (bad) report(status, 1);

  s_lo[t] = lo;
  s_hi[t] = hi;
  __syncthreads();
  for (int s = pow2_at_least(tpg) >> 1; s > 0; s >>= 1) {
    if (li < s && li + s < tpg) {
      s_lo[t] = fmin(s_lo[t], s_lo[t + s]);
      s_hi[t] = fmax(s_hi[t], s_hi[t + s]);
    }
    __syncthreads();
  }

  if (live && li == 0) {
    lo = s_lo[t];
    hi = s_hi[t];
    double step = 1.0;
    bool has_signal;
    if (MODE == QM_ASYM) {
      lo = fmin(lo, 0.0);
      hi = fmax(hi, 0.0);
      if (hi > lo) step = (hi - lo) / 15.0;
      has_signal = hi != lo;
    } else {
      const double amax = fmax(fabs(lo), fabs(hi));
      if (amax > 0.0) step = amax / (MODE == QM_F8 ? 448.0 : 7.0);
      has_signal = amax > 0.0;
    }
    float step_f = (float)step;
    // the host rounds in two steps; keep the compiler from folding the two
    // conversions into one FP64 -> FP16 rounding, which differs on ties
    asm volatile("" : "+v"(step_f));
    const _Float16 sh = (_Float16)step_f;
    const float sf = (float)sh;
    if (!(fabsf(sf) <= FLT_MAX) || (sf == 0.0f && has_signal)) report(status, 2);
    int zero = 8;
    if (MODE == QM_ASYM) {
      zero = clamp_code(round_half_away(-lo / (double)sf));
      atomicOr(zeros + row * (long long)words(G) + (g >> 3), (uint32_t)zero << (4 * (g & 7)));
    }
    scales[gid] = __builtin_bit_cast(uint16_t, sh);
    s_scale[lg] = sf;
    s_zero[lg] = zero;
  }
  __syncthreads();
  if (!live) return;

  const double sf = (double)s_scale[lg];
  const int zero = s_zero[lg];
  for (int wi = li; wi < nw; wi += tpg) {
    double v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int e = wi * 8 + j;
      v[j] = wi == li ? first[j] : (e < len ? (double)base[e] : 0.0);
    }
    if (MODE == QM_F8) {
      uint8_t* dst = q8 + row * (long long)K + k0 + wi * 8;
      uint32_t b[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) b[j] = encode_e4m3((float)(v[j] / sf));
      if (wi * 8 + 8 <= len && ((uintptr_t)dst & 7) == 0) {
        u2 out;
        out[0] = b[0] | (b[1] << 8) | (b[2] << 16) | (b[3] << 24);
        out[1] = b[4] | (b[5] << 8) | (b[6] << 16) | (b[7] << 24);
        *(u2*)dst = out;
      } else {
#pragma unroll
        for (int j = 0; j < 8; ++j)
          if (wi * 8 + j < len) dst[j] = (uint8_t)b[j];
      }
    } else {
      uint32_t word = 0;
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if (wi * 8 + j < len)
          word |= (uint32_t)clamp_code(round_half_away(v[j] / sf) + zero) << (4 * j);
      q32[row * (long long)words(K) + (k0 >> 3) + wi] = word;
    }
  }
}

// Arithmetic type of the elements.  FP64 sources divide in FP64 as the host does.  FP16 sources
// work in FP32 and multiply by the reciprocal: see quotient_code and quotient_magnitude.
template <typename T> struct Quot { typedef double type; };
template <> struct Quot<_Float16> { typedef float type; };

// clamp(round_half_away(v / sf) + zero, 0, 15) for FP16-representable v and sf > 0 without the
// division.  The quotient of two 11-bit significands is on a midpoint k + 1/2 or at least 2^-12 away from
// it, so a quotient that is made 2^-17 (relative) too large lands past the midpoint it was on,
// away from zero, and across no other: floor(q (1 + 2^-17) + zero + 1/2) is the code.  Its error (2^-22
// of q, 2^-20 from the sum) is below that shift from q = 1/2 on; beyond |q| = 16 every code
// saturates.  grown = (1 / sf) (1 + 2^-17).  Four instructions an element; the two tests of the
// remainder's sign around rint() that stood here before were fourteen.
__device__ __forceinline__ uint32_t quotient_code(float v, float grown, float zero_half) {
  return (uint32_t)__builtin_amdgcn_fmed3f(fmaf(v, grown, zero_half), 0.0f, 15.5f);
}

// Codes where the above does not hold: elements or steps that are not finite, a step of 0 (the group's
// extremum is below half of the smallest FP16 value times 7, 15 or 448).  rsf = 1 / sf.  A quotient
// of 64 or more or a NaN saturates, upwards unless v < 0.
__device__ __forceinline__ uint32_t quotient_code_any(float v, float sf, float rsf, int zero) {
  const float a = fabsf(v), t = fminf(a * rsf, 64.0f), c = rintf(t);
  int m = (int)c;  // round half up by the sign of |v| - (c -+ 1/2) sf
  if (fmaf(0.5f - c, sf, a) < 0.0f) --m;
  if (fmaf(-0.5f - c, sf, a) >= 0.0f) ++m;
  m = zero + (v < 0.0f ? -m : m);
  return (uint32_t)(m < 0 ? 0 : m > 15 ? 15 : m);
}

// The value of lane ^ m, m a power of two that is the same for all lanes.
__device__ __forceinline__ uint32_t lane_xor(uint32_t v, int m) {
  if (m == 1) return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0xB1, 0xF, 0xF, true);
  if (m == 2) return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x4E, 0xF, 0xF, true);
  return __shfl_xor(v, m);
}

typedef uint16_t us2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ void load8(const double* p, double v[8]) {
  typedef double d2 __attribute__((ext_vector_type(2)));
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const d2 x = ((const d2*)p)[i];
    v[2 * i] = x[0];
    v[2 * i + 1] = x[1];
  }
}
__device__ __forceinline__ void load8(const _Float16* p, float v[8]) {
  const h8 x = *(const h8*)p;
#pragma unroll
  for (int i = 0; i < 8; ++i) v[i] = (float)x[i];
}

// Whole rows of full groups whose word count is a power of two up to 64: a
// thread owns packed word `w` of the flattened (row, k) space, the gs / 8 lanes
// of a group combine their extrema with lane exchanges and every lane derives
// the group's scale itself -- no LDS round trip, fully coalesced 16-byte loads.
// Bound by vector instructions, not by memory: 8 slabs x 4096 x 128 FP16 keys and values (21.5 MB)
// took 10.1 us a call with some 220 of them a thread and 7.3 with 97 (E4M3 bytes 12.4 -> 8.4) while a launch of its
// own cleared the status word, and take 5.3 (6.5) now (3.5 at S = 16, which is the launch).
// ZPACK: zero-point words are assembled through LDS (G and the groups per workgroup both
// multiples of 8, or whole rows per workgroup: cache rows); otherwise nibbles are OR-ed in
// atomically, into words that a launch per side has cleared before (8 x 4096 x 128 with gs = 32:
// 13.6 us a call with those launches and FP64 divisions for step and zero-point, 9.2 without).
template <typename T, int MODE, bool ZPACK>
__global__ __launch_bounds__(QT) void quantize_rows_fast_kernel(
    const Sides<T> sd, long long nwords, int wpg, int wpg_shift, int G, const Status status) {
  begin_status(status);
  const T* __restrict__ src = sd.src[blockIdx.y];
  uint32_t* __restrict__ q32 = sd.q32[blockIdx.y];
  uint8_t* __restrict__ q8 = sd.q8[blockIdx.y];
  uint16_t* __restrict__ scales = sd.scales[blockIdx.y];
  uint32_t* __restrict__ zeros = sd.zeros[blockIdx.y];
  typedef typename Quot<T>::type A;
  __shared__ int s_zero[QT];
  const int t = threadIdx.x;
  const long long w = (long long)blockIdx.x * QT + t;
  const bool live = w < nwords;
  A v[8];
  A lo, hi;  // of the group; without zero-points of FP16 sources both are its largest magnitude
  bool special = false;  // FP16 sources: whether the wave has an element that is not finite
  if constexpr (sizeof(T) == 2) {
    // extrema on pairs of halves (whose minimum and maximum ignore a NaN); magnitudes as integers,
    // which NaN and infinity end up on top of
    u4 x = u4{0, 0, 0, 0};
    if (live) x = *(const u4*)(src + w * 8);
    us2 mag = __builtin_bit_cast(us2, x[0] & 0x7FFF7FFFu);
#pragma unroll
    for (int i = 1; i < 4; ++i)
      mag = __builtin_elementwise_max(mag, __builtin_bit_cast(us2, x[i] & 0x7FFF7FFFu));
    uint32_t top = mag[0] > mag[1] ? mag[0] : mag[1];
    // (a branch of the whole wave: as one of single lanes it cost 2 % of the kernel)
    special = __builtin_amdgcn_ballot_w64(top >= 0x7C00u) != 0;
    if (special) {
      if (top >= 0x7C00u) report(status, 1);
      top = 0;  // a NaN is no extremum: the scale is that of the group's other elements
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const uint32_t m = (x[i >> 1] >> (16 * (i & 1))) & 0x7FFFu;
        top = m > top && m <= 0x7C00u ? m : top;
      }
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = (A)__builtin_bit_cast(_Float16, (uint16_t)(x[j >> 1] >> (16 * (j & 1))));
    if constexpr (MODE == QM_ASYM) {
      // (minimum, -maximum) in one register
      h2 mn = as_h2(x[0]), mx = mn;
#pragma unroll
      for (int i = 1; i < 4; ++i) {
        mn = __builtin_elementwise_min(mn, as_h2(x[i]));
        mx = __builtin_elementwise_max(mx, as_h2(x[i]));
      }
      h2 ext = __builtin_elementwise_min(h2{mn[0], (_Float16)-mx[0]}, h2{mn[1], (_Float16)-mx[1]});
      for (int m = 1; m < wpg; m <<= 1) ext = __builtin_elementwise_min(ext, as_h2(lane_xor(as_u32(ext), m)));
      lo = (A)ext[0];
      hi = -(A)ext[1];
    } else {
      for (int m = 1; m < wpg; m <<= 1) {
        const uint32_t o = lane_xor(top, m);
        top = o > top ? o : top;
      }
      lo = hi = (A)__builtin_bit_cast(_Float16, (uint16_t)top);
    }
  } else {
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = (A)0;
    if (live) load8(src + w * 8, v);
    lo = hi = v[0];
    bool bad = false;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      bad |= !(fabs((double)v[j]) <= DBL_MAX);
      lo = v[j] < lo ? v[j] : lo;
      hi = v[j] > hi ? v[j] : hi;
    }
    if (bad) report(status, 1);
    for (int m = 1; m < wpg; m <<= 1) {
      const A olo = __shfl_xor(lo, m), ohi = __shfl_xor(hi, m);
      lo = olo < lo ? olo : lo;
      hi = ohi > hi ? ohi : hi;
    }
  }
  // Scale of the group, in every lane.  The step goes FP64 -> FP32 -> FP16 on the
  // host.  For FP16 sources without zero-points the FP32 step is amax / 7 (/ 448)
  // of an 11-bit amax: its binary expansion is periodic with period 3, so it is
  // never within an FP64 rounding error of an FP32 midpoint and one correctly
  // rounded FP32 division gives the same FP32 value as the two-step rounding.
  float step_f;
  bool has_signal;
  double dlo = (double)lo, dhi = (double)hi;
  if (MODE == QM_ASYM) {
    dlo = fmin(dlo, 0.0);
    dhi = fmax(dhi, 0.0);
    const double range = dhi - dlo;
    double step;
    if constexpr (sizeof(T) == 2) {
      // range / 15, correctly rounded: a quotient by the rounded reciprocal, corrected once by its
      // residual (a finite range is between 2^-24 and 2^17, so nothing under- or overflows; an
      // infinite one leaves NaN, and the minimum turns that into a step past FP16's range)
      const double q = range * (1.0 / 15.0);
      step = fmin(fma(fma(-q, 15.0, range), 1.0 / 15.0, q), DBL_MAX);
    } else {
      step = range / 15.0;
    }
    step_f = (float)(range > 0.0 ? step : 1.0);
    has_signal = dhi != dlo;
  } else if (sizeof(T) == 2) {
    const float amax = (float)hi;
    step_f = amax > 0.0f ? amax / (MODE == QM_F8 ? 448.0f : 7.0f) : 1.0f;
    has_signal = amax > 0.0f;
  } else {
    const double amax = fmax(fabs(dlo), fabs(dhi));
    step_f = (float)(amax > 0.0 ? amax / (MODE == QM_F8 ? 448.0 : 7.0) : 1.0);
    has_signal = amax > 0.0;
  }
  asm volatile("" : "+v"(step_f));  // keep the FP32 and FP16 roundings separate
  const _Float16 sh = (_Float16)step_f;
  const float sf = (float)sh;
  int zero = 8;
  const float grown = __builtin_amdgcn_rcpf(sf) * (1.0f + 0x1p-17f);
  if constexpr (MODE == QM_ASYM) {
    if constexpr (sizeof(T) == 2) zero = (int)quotient_code(-(float)dlo, grown, 0.5f);
    else zero = clamp_code(round_half_away(-dlo / (double)sf));
  }
  const bool leader = live && (t & (wpg - 1)) == 0;
  const long long gid = w >> wpg_shift;
  if (leader) {
    if (!(fabsf(sf) <= FLT_MAX) || (sf == 0.0f && has_signal)) report(status, 2);
    scales[gid] = __builtin_bit_cast(uint16_t, sh);
    if (MODE == QM_ASYM && !ZPACK) {
      const long long row = gid / G;
      const int g = (int)(gid - row * G);
      atomicOr(zeros + row * (long long)words(G) + (g >> 3), (uint32_t)zero << (4 * (g & 7)));
    }
  }
  if (MODE == QM_ASYM && ZPACK) {
    if ((t & (wpg - 1)) == 0) s_zero[t >> wpg_shift] = zero;
    __syncthreads();
    const int gpb = QT >> wpg_shift;
    if ((G & 7) == 0) {
      const long long zw = ((long long)blockIdx.x * gpb >> 3) + t;
      if (t < (gpb >> 3) && zw * 8 * wpg < nwords) {
        uint32_t word = 0;
#pragma unroll
        for (int j = 0; j < 8; ++j) word |= (uint32_t)s_zero[t * 8 + j] << (4 * j);
        zeros[zw] = word;
      }
    } else {  // whole rows per workgroup: thread t makes word t of them
      const int wpr = (G + 7) >> 3, r = t / wpr, i = t - r * wpr;
      const long long row = (long long)blockIdx.x * (gpb / G) + r;
      if (r < gpb / G && row * G * wpg < nwords) {
        uint32_t word = 0;
        for (int g = 8 * i; g < min(8 * i + 8, G); ++g) word |= (uint32_t)s_zero[r * G + g] << (4 * (g & 7));
        zeros[row * wpr + i] = word;
      }
    }
  }
  if constexpr (sizeof(T) == 2) {
    // (elements are read again: kept for this path, their registers cost the other one 3 %)
    const bool plain = __builtin_amdgcn_classf(sf, 0x100);  // positive and finite
    if (special || __builtin_amdgcn_ballot_w64(!plain) != 0) {
      if (!live) return;
      const float rsf = __builtin_amdgcn_rcpf(sf);
      float u[8];
      load8(src + w * 8, u);
      u2 out = u2{0, 0};
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        if (MODE == QM_F8) {  // NaN is 0x7F; a step of 0 or infinity leaves no residual to correct by
          const float x = u[j] * rsf;
          out[j >> 2] |= encode_e4m3(plain ? copysignf(quotient_magnitude(u[j], sf, rsf), x) : x) << (8 * (j & 3));
        } else {
          out[0] |= quotient_code_any(u[j], sf, rsf, zero) << (4 * j);
        }
      }
      if (MODE == QM_F8) *(u2*)(q8 + w * 8) = out;
      else q32[w] = out[0];
      return;
    }
  }
  if (!live) return;
  const A sfa = (A)sf;
  if (MODE == QM_F8) {
    u2 out;
    if constexpr (sizeof(T) == 2) {
      const float rsf = __builtin_amdgcn_rcpf(sf);
      float mag[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) mag[j] = quotient_magnitude(v[j], sf, rsf);
      out[0] = pack_e4m3(mag, v);
      out[1] = pack_e4m3(mag + 4, v + 4);
    } else {
      uint32_t b[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) b[j] = encode_e4m3((float)(v[j] / sfa));
      out[0] = b[0] | (b[1] << 8) | (b[2] << 16) | (b[3] << 24);
      out[1] = b[4] | (b[5] << 8) | (b[6] << 16) | (b[7] << 24);
    }
    *(u2*)(q8 + w * 8) = out;
  } else {
    uint32_t word = 0;
    const float zero_half = (float)zero + 0.5f;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      if constexpr (sizeof(T) == 2) {
        word |= quotient_code(v[j], grown, zero_half) << (4 * j);
      } else {
        const int c = (int)round_half_away(v[j] / sfa) + zero;
        word |= (uint32_t)(c < 0 ? 0 : (c > 15 ? 15 : c)) << (4 * j);
      }
    }
    q32[w] = word;
  }
}

// mx.hpp:91-101 in closed form: the smallest e with amax <= TOP * 2^e, TOP the
// largest magnitude of the element type (6 for E2M1, 448 for E4M3).  With amax in
// [2^p, 2^(p+1)) the answer lies within two steps of p - ilogb(TOP).
template <int TOP>
__device__ __forceinline__ int mx_exponent(double amax, bool* out_of_range) {
  if (!(amax > 0.0)) return 0;
  if (amax <= (double)TOP * 0x1p-127) return -127;
  const int p = (int)((__builtin_bit_cast(uint64_t, amax) >> 52) & 0x7FFu) - 1023;
  int e = p - (TOP == 6 ? 2 : 9);  // TOP * 2^(e - 1) < 2^p <= amax
  if (amax > (double)TOP * ldexp(1.0, e)) ++e;
  if (amax > (double)TOP * ldexp(1.0, e)) ++e;
  if (e > 127) {
    *out_of_range = true;
    e = 127;
  }
  return e;
}

// The same from the FP32 value of a finite FP16 maximum: TOP is 1.5 * 2^2 or 1.75 * 2^8, so e is
// p - 2 (p - 8), and one more where the significand is past TOP's.  (e is -32 .. 14: in range.)
template <int TOP>
__device__ __forceinline__ int mx_exponent_f16(float amax) {
  const uint32_t b = __builtin_bit_cast(uint32_t, amax);
  return amax > 0.0f ? (int)((b + (TOP == 6 ? 0x3FFFFFu : 0x1FFFFFu)) >> 23) - (TOP == 6 ? 129 : 135) : 0;
}

// mx.hpp:103-108: index of the nearest E2M1 magnitude, the lower one on ties.
__device__ __forceinline__ int nearest_e2m1(double a) {
  const double mags[8] = {0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0};
  int best = 0;
  double dbest = a;
#pragma unroll
  for (int i = 1; i < 8; ++i) {
    const double d = __builtin_elementwise_abs(mags[i] - a);
    if (d < dbest) {
      best = i;
      dbest = d;
    }
  }
  return best;
}

// The packed word of eight scaled FP16 values, at most 6 in magnitude.  The hardware conversion
// rounds to nearest even; values made 2^-14 (relative) smaller leave a tie towards zero, and
// pass no other: with 11 significant bits a value is on a tie or 2^-11 (relative) past it.
__device__ __forceinline__ uint32_t pack_e2m1(const float* u) {
  constexpr float SHRINK = 1.0f - 0x1p-14f;
  uint32_t w = 0;
  w = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(w, u[0] * SHRINK, u[1] * SHRINK, 1.0f, 0);
  w = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(w, u[2] * SHRINK, u[3] * SHRINK, 1.0f, 1);
  w = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(w, u[4] * SHRINK, u[5] * SHRINK, 1.0f, 2);
  return __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(w, u[6] * SHRINK, u[7] * SHRINK, 1.0f, 3);
}

// Four threads per 32-element block, eight elements each: one packed word of
// E2M1 codes, or (F8: the MXFP8 activation format, no host counterpart in the
// reference; same block rule with 448 in place of 6) eight E4M3 bytes.  FP16 sources
// were bound by vector instructions (seven compares and selects a code, the exponent in FP64):
// 2048 x 4096 took 12.7 us a call into MXFP4 and 12.0 into MXFP8, 6.4 and 7.0 with the hardware conversions and
// the exponent from integer arithmetic, and takes 5.0 and 5.7 since the status word has no launch of its own (16 rows: 3.3).
template <typename T, bool FULL, bool F8>
__global__ __launch_bounds__(QT) void quantize_mx_kernel(const T* __restrict__ src,
                                                         long long rows, int K, int B,
                                                         uint32_t* __restrict__ q,
                                                         uint8_t* __restrict__ q8,
                                                         uint8_t* __restrict__ scales,
                                                         const Status status) {
  begin_status(status);
  const long long id = (long long)blockIdx.x * QT + threadIdx.x;
  const long long blk = id >> 2;
  const int j4 = (int)(id & 3);
  const bool live = blk < rows * B;
  long long row = 0;
  int b = 0;
  if (live) {
    row = blk / B;
    b = (int)(blk - row * B);
  }
  const int k0 = b * 32 + j4 * 8;
  const int n = live ? (K - k0 < 0 ? 0 : (K - k0 > 8 ? 8 : K - k0)) : 0;
  const T* base = src + row * (long long)K + k0;
  // FP16 sources work in FP32: scaling by a power of two is exact, and so is
  // everything the encoders do with an 11-bit significand
  typedef typename Quot<T>::type A;
  A v[8];
  if constexpr (FULL) {  // K a multiple of 8 and 16-byte aligned rows: four 16-byte loads
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = (A)0;
    if (n) load8(base, v);
  } else {
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = j < n ? (A)base[j] : (A)0;
  }
  int e;
  bool bad = false;
  if constexpr (sizeof(T) == 2) {
    // the largest magnitude as an integer, which NaN and infinity end up on top of
    uint32_t top = 0;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const uint32_t mag = __builtin_bit_cast(uint32_t, v[j]) & 0x7FFFFFFFu;
      top = mag > top ? mag : top;
    }
    bad = top >= 0x7F800000u;
    if (bad) {  // a NaN is no maximum: the exponent is that of the block's other elements
      report(status, 1);
      top = 0;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const uint32_t mag = __builtin_bit_cast(uint32_t, v[j]) & 0x7FFFFFFFu;
        top = mag > top && mag <= 0x7F800000u ? mag : top;
      }
    }
    const uint32_t o1 = lane_xor(top, 1);
    top = o1 > top ? o1 : top;
    const uint32_t o2 = lane_xor(top, 2);
    top = o2 > top ? o2 : top;
    e = mx_exponent_f16<F8 ? 448 : 6>(__builtin_bit_cast(float, top));
    if (top == 0x7F800000u) {
      e = 127;
      if (j4 == 0) report(status, 2);
    }
  } else {
    A amax = (A)0;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const A av = v[j] < (A)0 ? -v[j] : v[j];
      bad |= !(av <= (A)DBL_MAX);
      amax = av > amax ? av : amax;
    }
    if (bad) report(status, 1);
    const A o1 = __shfl_xor(amax, 1);
    amax = o1 > amax ? o1 : amax;
    const A o2 = __shfl_xor(amax, 2);
    amax = o2 > amax ? o2 : amax;
    bool range = false;
    e = mx_exponent<F8 ? 448 : 6>((double)amax, &range);
    if (range && j4 == 0) report(status, 2);
  }
  if (n == 0) return;
  A u[8];  // v / 2^e
  if constexpr (sizeof(T) == 2) {
#pragma unroll
    for (int j = 0; j < 8; ++j) u[j] = ldexpf(v[j], -e);
  } else {
    // |e| <= 127, so 2^-e is a normal double and v * 2^-e is the same real number
    // as v / 2^e, rounded the same way: the host's quotient without the division
    const double inv = ldexp(1.0, -e);
#pragma unroll
    for (int j = 0; j < 8; ++j) u[j] = v[j] * inv;
  }
  if (F8) {
    uint8_t* dst = q8 + row * (long long)K + k0;
    float val[8], mag[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) val[j] = (float)u[j], mag[j] = fabsf(val[j]);
    u2 out = u2{pack_e4m3(mag, val), pack_e4m3(mag + 4, val + 4)};
    if (bad) {  // NaN is 0x7F
      out = u2{0, 0};
#pragma unroll
      for (int j = 0; j < 8; ++j) out[j >> 2] |= encode_e4m3(val[j]) << (8 * (j & 3));
    }
    if (n == 8 && ((uintptr_t)dst & 7) == 0) {
      *(u2*)dst = out;
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if (j < n) dst[j] = (uint8_t)(out[j >> 2] >> (8 * (j & 3)));
    }
  } else {
    uint32_t word = 0;
    if constexpr (sizeof(T) == 2) {
      if (bad) {  // E2M1 has no code for them: zeros, as from FP64 sources
#pragma unroll
        for (int j = 0; j < 8; ++j) u[j] = fabsf(u[j]) < INFINITY ? u[j] : copysignf(0.0f, u[j]);
      }
      word = pack_e2m1(u);  // (elements past the row are +0: code 0)
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if (j < n) {
          const uint32_t code = (__builtin_signbit(u[j]) ? 8u : 0u) |
                                (uint32_t)nearest_e2m1(u[j] < (A)0 ? -u[j] : u[j]);
          word |= code << (4 * j);
        }
    }
    q[row * (long long)words(K) + b * 4 + j4] = word;
  }
  if (j4 == 0) scales[blk] = (uint8_t)(e + 127);
}

template <typename T, int MODE>
hipError_t launch_rows_t(const Sides<T>& sd, int nsides, long long rows, int K, int gs,
                         const Status& status, hipStream_t s) {
  const int G = (K + gs - 1) / gs;
  const int wpg = gs >> 3, tpg = wpg < QT ? wpg : QT, gpb = QT / tpg;
  const bool pow2 = (wpg & (wpg - 1)) == 0;
  bool aligned = true;
  for (int i = 0; i < nsides; ++i)
    aligned = aligned && ((uintptr_t)sd.src[i] & 15) == 0 &&
              (MODE != QM_F8 || ((uintptr_t)sd.q8[i] & 7) == 0);
  const bool fast = pow2 && wpg <= 64 && K % gs == 0 && aligned;
  // (a workgroup covers 2048 elements; with whole rows a row has at most one word per thread)
  const bool zpack = fast && MODE == QM_ASYM && ((G % 8 == 0 && (QT / wpg) % 8 == 0) || (QT * 8) % K == 0);
  if (MODE == QM_ASYM && !zpack) {
    // zero-points are OR-ed in nibble by nibble
    const long long nz = rows * words(G);
    for (int i = 0; i < nsides; ++i)
      fill_words_kernel<<<dim3((unsigned)((nz + 255) / 256)), dim3(256), 0, s>>>(sd.zeros[i], nz, 0u);
  }
  if (fast) {
    const long long nwords = rows * (K >> 3);
    const long long nb = (nwords + QT - 1) / QT;
    if (nb > 0x7FFFFFFFLL) return hipErrorInvalidConfiguration;
    const int shift = __builtin_ctz(wpg);
    const dim3 grid((unsigned)nb, (unsigned)nsides);
    if (zpack)
      quantize_rows_fast_kernel<T, MODE, true><<<grid, dim3(QT), 0, s>>>(sd, nwords, wpg, shift, G,
                                                                        status);
    else
      quantize_rows_fast_kernel<T, MODE, false><<<grid, dim3(QT), 0, s>>>(sd, nwords, wpg, shift,
                                                                         G, status);
    return hipGetLastError();
  }
  const long long blocks = (rows * G + gpb - 1) / gpb;
  if (blocks > 0x7FFFFFFFLL) return hipErrorInvalidConfiguration;
  quantize_rows_kernel<T, MODE><<<dim3((unsigned)blocks, (unsigned)nsides), dim3(QT), 0, s>>>(
      sd, rows, K, gs, G, status);
  return hipGetLastError();
}

template <typename T>
hipError_t launch_rows(int mode, const QuantSide* sides, int nsides, long long rows, int K, int gs,
                       const Status& status, hipStream_t s) {
  Sides<T> sd{};
  for (int i = 0; i < nsides; ++i) {
    sd.src[i] = (const T*)sides[i].src;
    sd.q32[i] = sides[i].q32;
    sd.q8[i] = sides[i].q8;
    sd.scales[i] = sides[i].scales;
    sd.zeros[i] = sides[i].zeros;
  }
  if (mode == QM_SYM) return launch_rows_t<T, QM_SYM>(sd, nsides, rows, K, gs, status, s);
  if (mode == QM_ASYM) return launch_rows_t<T, QM_ASYM>(sd, nsides, rows, K, gs, status, s);
  return launch_rows_t<T, QM_F8>(sd, nsides, rows, K, gs, status, s);
}

// The status word of one call, from its ticket to the launch.
//
// Calls get a slot by the stream they are on, so that only calls that run one after the other share
// one; the slot's lock is held until the kernel is enqueued, so that threads that use one stream enqueue
// in the order of their tickets.  A slot stays its stream's (a stream created later at the same
// address goes on with its tickets).  A launch of its own clears the word, and the ticket is 0, where
// that cannot be had: in a stream that is being captured (a replay would find its ticket from the replay
// before; the legacy stream cannot be captured), for the handles that stand for the legacy and the
// calling thread's stream, and for streams past the first QZ_SLOTS.
class StatusCall {
 public:
  hipError_t begin(int* word, hipStream_t s) {
    st_ = Status{word, 0};
    if (Slot* const slot = slot_of(s)) {
      held_ = std::unique_lock<std::mutex>(slot->lock);
      st_.ticket = ++slot->calls * QZ_SLOTS + (qz_ticket)(slot - slots);
      return hipSuccess;
    }
    fill_words_kernel<<<dim3(1), dim3(64), 0, s>>>((uint32_t*)word, 1, 0u);
    return hipGetLastError();
  }
  const Status& status() const { return st_; }

 private:
  struct Slot {
    std::mutex lock;  // of calls
    qz_ticket calls = 0;
    int dev = -1;
    hipStream_t stream = nullptr;
  };
  static Slot slots[QZ_SLOTS];

  static Slot* slot_of(hipStream_t s) {
    int dev = 0;
    if (s == hipStreamLegacy || s == hipStreamPerThread || hipGetDevice(&dev) != hipSuccess) return nullptr;
    if (s != nullptr) {
      hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
      if (hipStreamIsCapturing(s, &cap) != hipSuccess) return (void)hipGetLastError(), nullptr;
      if (cap != hipStreamCaptureStatusNone) return nullptr;
    }
    static std::mutex table;  // of dev and stream of all slots
    static int used = 0;
    const std::lock_guard<std::mutex> guard(table);
    for (int i = 0; i < used; ++i)
      if (slots[i].stream == s && slots[i].dev == dev) return &slots[i];
    if (used == QZ_SLOTS) return nullptr;
    slots[used].dev = dev, slots[used].stream = s;
    return &slots[used++];
  }

  Status st_{};
  std::unique_lock<std::mutex> held_;
};
StatusCall::Slot StatusCall::slots[QZ_SLOTS];

}  // namespace

hipError_t launch_quantize_rows(int mode, const QuantSide* sides, int nsides, int src_f16,
                                long long rows, int K, int gs, int* word, hipStream_t s) {
  StatusCall call;
  if (hipError_t e = call.begin(word, s); e != hipSuccess) return e;
  const Status& status = call.status();
  return src_f16 ? launch_rows<_Float16>(mode, sides, nsides, rows, K, gs, status, s)
                 : launch_rows<double>(mode, sides, nsides, rows, K, gs, status, s);
}

hipError_t launch_quantize_mx(const void* src, int src_f16, long long rows, int K, uint32_t* q,
                              uint8_t* scales, int* word, hipStream_t s) {
  const int B = (K + 31) / 32;
  const long long blocks = (rows * B * 4 + QT - 1) / QT;
  if (blocks > 0x7FFFFFFFLL) return hipErrorInvalidConfiguration;
  StatusCall call;
  if (hipError_t e = call.begin(word, s); e != hipSuccess) return e;
  const Status& status = call.status();
  const dim3 grid((unsigned)blocks), block(QT);
  const bool vec = K % 8 == 0 && ((uintptr_t)src & 15) == 0;
  if (src_f16 && vec)
    quantize_mx_kernel<_Float16, true, false><<<grid, block, 0, s>>>((const _Float16*)src, rows, K,
                                                                    B, q, nullptr, scales, status);
  else if (src_f16)
    quantize_mx_kernel<_Float16, false, false><<<grid, block, 0, s>>>((const _Float16*)src, rows, K,
                                                                     B, q, nullptr, scales, status);
  else if (K % 8 == 0 && ((uintptr_t)src & 15) == 0)
    quantize_mx_kernel<double, true, false><<<grid, block, 0, s>>>((const double*)src, rows, K, B,
                                                                  q, nullptr, scales, status);
  else
    quantize_mx_kernel<double, false, false><<<grid, block, 0, s>>>((const double*)src, rows, K, B,
                                                                   q, nullptr, scales, status);
  return hipGetLastError();
}

hipError_t launch_quantize_mx8(const void* src, int src_f16, long long rows, int K, uint8_t* q,
                               uint8_t* scales, int* word, hipStream_t s) {
  const int B = (K + 31) / 32;
  const long long blocks = (rows * B * 4 + QT - 1) / QT;
  if (blocks > 0x7FFFFFFFLL) return hipErrorInvalidConfiguration;
  StatusCall call;
  if (hipError_t e = call.begin(word, s); e != hipSuccess) return e;
  const Status& status = call.status();
  const dim3 grid((unsigned)blocks), block(QT);
  if (src_f16 && K % 8 == 0 && ((uintptr_t)src & 15) == 0)
    quantize_mx_kernel<_Float16, true, true><<<grid, block, 0, s>>>((const _Float16*)src, rows, K,
                                                                   B, nullptr, q, scales, status);
  else if (src_f16)
    quantize_mx_kernel<_Float16, false, true><<<grid, block, 0, s>>>((const _Float16*)src, rows, K,
                                                                    B, nullptr, q, scales, status);
  else
    quantize_mx_kernel<double, false, true><<<grid, block, 0, s>>>((const double*)src, rows, K, B,
                                                                  nullptr, q, scales, status);
  return hipGetLastError();
}

}  // namespace w4k
