// Launch functions of the gfx950 kernels (one per kernel family).  They take
// already-validated arguments and only enqueue work on `stream`.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/w4_abi.h"

namespace w4k {

// Which packed format a weight view carries.
struct WView {
  int mx;  // 0: W4 affine (scales FP16, optional zero-points), 1: MXFP4
  int N, K;
  int gs, G, symmetric;  // W4 only
  int B;                 // MX only
  const uint32_t* q;
  const void* scales;  // w4_half* (W4) or uint8_t* (MX)
  const uint32_t* zeros;
};

inline WView view_of(const w4_packed_view& p) {
  return WView{0, p.N, p.K, p.gs, p.G, p.symmetric, 0, p.q, p.scales, p.zeros};
}
inline WView view_of(const w4_packed_mx_view& p) {
  return WView{1, p.N, p.K, 32, p.B, 1, p.B, p.q, p.scales, nullptr};
}

// Compute units of the current device (kept per device); 0 on error.
int device_cus();

// dequant.hip
hipError_t launch_dequant(const WView& v, w4_half* w, hipStream_t s);
hipError_t launch_dequant_f8(const uint8_t* q, const w4_half* sc, w4_half* w,
                             int S, int D, int gs, hipStream_t s);

// gemm_simt.hip
hipError_t launch_gemm_simt(const WView& v, const w4_half* x, w4_half* c, int M,
                            hipStream_t s, w4_half* w_out);
// gemm_mfma.hip
hipError_t launch_gemm_mfma(const WView& v, const w4_half* x, w4_half* c, int M,
                            hipStream_t s, w4_half* w_out);
// Which kernel it takes, without a hook, for operands aligned to 16 bytes: see w4_gemm_plan_for.
int gemm_plan(const WView& v, int M);

// gemm_tile_dma.hip: large-M W4 kernel with direct-to-LDS operand loads; false
// (nothing launched) when the arguments are not its shape.
bool try_tile_dma(const WView& v, const w4_half* x, w4_half* c, int M, hipStream_t s,
                  w4_half* w_out, hipError_t* err);

// gemm_tile256.hip: the same scheme on 256 x 256 tiles, for try_tile_dma to hand unhooked
// calls to once it has checked the operands; false (nothing launched) when that tile
// would not at least halve the rounds of workgroups on `cus` compute units.
bool try_tile256(const WView& v, const w4_half* x, w4_half* c, int M, hipStream_t s, int cus,
                 hipError_t* err);

// gemm_block.hip: middle M (17 to some hundred rows, at long K from 3 on; from 5 for sizes that are not whole), blocks
// of W and x as square as few rounds of workgroups allow, hooked calls included; false (nothing launched) when another
// kernel is ahead.
bool try_block(const WView& v, const w4_half* x, w4_half* c, int M, hipStream_t s, w4_half* w_out,
               int shape, hipError_t* err);
// shape: the block that any_plan() names, or -1: block_plan()'s own.
// Its block for operands aligned to 16 bytes: 10 x tiles of W + row tiles of x; 0: not its shape.
int block_shape(const WView& v, int M);

// Time of its best block in units of 10 ns, and which; -1: none.  block_plan_time: for shapes of whole tiles, chunks and
// groups, where another kernel may be ahead as well; block_any_time: for every other.
int block_plan_time(const WView& v, int M, int* time);
int block_any_time(const WView& v, int M, int cus, int* time);

// gemm_tile_any.hip: the kernel of gemm_tile_dma.hip for any group size and any K that are multiples of 8, and the
// plan for calls whose sizes the kernels for whole tiles, chunks and groups do not take: kind 1 a block
// (shape: its index), 2 a tile, 0 another kernel, 3 another kernel and no block (block_plan() has been asked).
struct AnyPlan {
  int kind, shape;
};
AnyPlan any_plan(const WView& v, int M);
// Whether a reciprocal gives the group of every word (see launch() in tile_dma.cuh).
bool any_group_fits(const WView& v);
// Launches the planned tile; false (nothing launched) when the arrays are not aligned for it.
bool try_tile_any(const WView& v, const w4_half* x, w4_half* c, int M, hipStream_t s, w4_half* w_out, int shape,
                  hipError_t* err);

// gemm_decode_resident.hip: M <= 64 with the activations fetched once per workgroup
// (several 16-row tiles each).  Same order of additions as the K-split decode
// kernels of gemm_mfma.hip, which serve the hooked calls of these shapes.
bool decode_resident_applies(const WView& v, const w4_half* x, const w4_half* c, int M);
hipError_t launch_decode_resident(const WView& v, const w4_half* x, w4_half* c, int M,
                                  hipStream_t s);
// Long K (8, 11 or 14 chunks of 128 k per wave) with more than 12 to 16 activation rows on a grid of
// more tiles than compute units: the resident kernel then gives a workgroup two tiles, and the
// long-K kernel below leaves the shape to it.
bool decode_resident_shares_long_k(const WView& v, const w4_half* x, const w4_half* c, int M);

// gemm_decode_longk.hip: M <= 64 at long K (5 to 16 chunks of 128 k per wave; 2 to 4 on thin grids), one
// 16-row tile per workgroup with activations and codes requested chunk by chunk while
// earlier chunks multiply; same order of additions as the two kernels above.
bool decode_longk_applies(const WView& v, const w4_half* x, const w4_half* c, int M);
hipError_t launch_decode_longk(const WView& v, const w4_half* x, w4_half* c, int M,
                               hipStream_t s);

// gemm_decode_general.hip: M <= 64 for any group size (multiple of 8) and any K % 8 == 0
// with 1024 < K <= 5120, group parameters through LDS; same order of additions as the
// K-split decode kernels of gemm_mfma.hip.
bool decode_general_applies(const WView& v, const w4_half* x, const w4_half* c, int M);
// Tiles of W per workgroup of that kernel; 0: not its arguments.
int decode_general_tiles(const WView& v, int M);
hipError_t launch_decode_general(const WView& v, const w4_half* x, w4_half* c, int M,
                                 hipStream_t s);

// flash.hip -- one description for the four cache kinds
struct FlashArgs {
  int kind;  // 0 FP16, 1 W4, 2 FP8
  int H;     // cache slabs addressed by a (sequence, kv-head) pair: nseq * Hkv
  int S, D, gs, G, symmetric;
  int group;       // query heads per slab
  int scale_mode;  // FP8: 0 per (row, group), 1 per slab
  const void* k;   // FP16: halves; W4: packed words; FP8: bytes
  const void* v;
  const w4_half* s_k;
  const w4_half* s_v;
  const uint32_t* z_k;
  const uint32_t* z_v;
  // paging (W4 only): bt == nullptr means contiguous slabs of S rows
  const int* bt;
  int bt_stride;   // entries per sequence table
  int page, pool_rows;
  int Hkv;         // paged: pool slabs; sequence = slab / Hkv
  int scratch_id;  // which of the FL_SCRATCH_IDS buffers holds the partials
  const w4_half* q;
  w4_half* out;
  w4_half* k_out;
  w4_half* v_out;
};
// Scratch buffers that calls in flight may be using: 0 the fixed one; from 1 on the grown one and
// those it has replaced, by the logarithm of their size (each is at least twice its predecessor).
constexpr int FL_SCRATCH_IDS = 32;
enum { KIND_F16 = 0, KIND_W4 = 1, KIND_F8 = 2 };  // FlashArgs::kind

// Split of the sequence over workgroups (shared by both phase-1 kernels).
constexpr int FL_DIRECT_MAX_S = 512;  // longest cache that always has one split per slab (matrix-core kernel)
constexpr int FL_DIRECT_MIN_H = 512;  // number of slabs from which on every cache has
struct FlashPlan {
  int split_len, nsplit;
};
FlashPlan flash_plan(const FlashArgs& a);
// flash_mfma.hip: whether the matrix-core phase 1 (D = 128) takes these arguments.
bool flash_mfma_applies(const FlashArgs& a);
// Whether its last workgroup of every slab merges the splits itself (no second launch).
bool flash_merges_in_place(const FlashArgs& a, const FlashPlan& pl);
// Whether its tiles go through LDS (else through registers).
bool flash_tiles_in_lds(const FlashArgs& a, const FlashPlan& pl);
// Launches it; false when the arguments need the general kernel (nothing is
// launched then).
bool try_flash_mfma(const FlashArgs& a, const FlashPlan& pl, float* part, hipStream_t s,
                    hipError_t* err);

// Floats of scratch the split-S partials need for these arguments.
size_t flash_scratch_floats(const FlashArgs& a);
hipError_t launch_flash(const FlashArgs& a, float* scratch, hipStream_t s);

// quantize.hip -- the host quantizers as kernels.  mode: 0 W4 symmetric, 1 W4 with
// zero-points, 2 E4M3 bytes; src is FP64 or (src_f16) FP16; `rows` rows of K
// elements, groups of gs along K.  status: cleared by the call, then bit 0
// non-finite input, bit 1 scale out of range.
struct QuantSide {  // one source and its outputs (q32: W4 words, q8: E4M3 bytes)
  const void* src;
  uint32_t* q32;
  uint8_t* q8;
  w4_half* scales;
  uint32_t* zeros;
};
// nsides (1 or 2) jobs of the same shape in one launch: the K and V sides of a cache
hipError_t launch_quantize_rows(int mode, const QuantSide* sides, int nsides, int src_f16,
                                long long rows, int K, int gs, int* status, hipStream_t s);
hipError_t launch_quantize_mx(const void* src, int src_f16, long long rows, int K, uint32_t* q,
                              uint8_t* scales, int* status, hipStream_t s);
// gemm_mxnative.hip -- both operands packed MXFP4 (x.N = M rows of K), scaled MFMA
hipError_t launch_gemm_mx_w4a4(const w4_packed_mx_view& w, const w4_packed_mx_view& x,
                               w4_half* c, hipStream_t s);
hipError_t launch_gemm_mx_w4a8(const w4_packed_mx_view& w, const w4_act_mx8_view& x, w4_half* c,
                               hipStream_t s);
// Which kernel they take with arrays aligned to 16 bytes (x8: E4M3 activations): see w4_gemm_mx_plan_for.
int mx_plan(bool x8, int M, int N, int K);
hipError_t launch_quantize_mx8(const void* src, int src_f16, long long rows, int K, uint8_t* q,
                               uint8_t* scales, int* status, hipStream_t s);

}  // namespace w4k
