// The W3 weight stream on gfx950: dense linear and routed-expert grouped GEMMs for decode / verify sized calls.
//
// One wavefront owns a block column of the tile layout: 64 output rows x a range of 128-k chunks, for one "slot" of up
// to 16 activation rows. A chunk is a contiguous 3328-byte block (packed codes, then scales); it travels from memory
// into the wavefront's ring in LDS without passing through registers, two chunks ahead of the one being expanded.
// The expansion happens in registers (v_perm_b32 over the 8-byte E4M3 codebook, then the hardware FP8 -> BF16 pair
// conversion: exact) and feeds sixteen v_mfma_f32_16x16x32_bf16 (4 row tiles x 4 scale groups): one MFMA is exactly
// one 32-group, so the group scale is folded into the FP32 accumulator after it (acc += part * scale), as the
// reference kernel does per group (hibana/kernels/csrc/w3_gemm.cu:105-108); the FP32 row scale is applied in the
// epilogue (:209-210). Activations are BF16, read straight from global memory (they stay in L2) as the MFMA A operand.
// Slots of at most four rows (most of a decode or verify step) take a second body that packs the four groups into the
// idle MFMA rows and so folds a quarter of the scales. The wavefronts of a workgroup split K (partials reduced through
// LDS in a fixed order) and/or take neighbouring 64-row blocks. No atomics on floating point anywhere: results are
// bitwise repeatable.
//
// Calls of more than sixteen rows, and routed ones with many rows an expert (prefill), go to the panel kernel of
// panel_kernel.hpp instead, through the TileW3 policies below; hb_tune("w3_tile", 1 | 2) forces one or the other.
#include <string.h>

#include <algorithm>
#include <atomic>
#include <mutex>
#include <type_traits>

#include "panel_kernel.hpp"
#include "ring.hpp"
#include "route.hpp"
#include "stream_common.hpp"
#include "w3_layout.hpp"

namespace hb {

struct Chunk {  // the weight side of one 64-row x 128-k block
  u32x4_t w0, w1, w2, sc;
};

struct Chunk2 {  // the same of a two-bit matrix: eight code dwords a lane
  u32x4_t w0, w1, sc;
};

// The eight selectors of 16-row tile NT of a chunk, and the dword of its four scale bytes.
template <int NT>
__device__ __forceinline__ void chunk_selectors(const Chunk& ch, uint32_t sel[8]) {
  if (NT == 0) w3_selectors(ch.w0.x, ch.w0.y, ch.w0.z, sel);
  if (NT == 1) w3_selectors(ch.w0.w, ch.w1.x, ch.w1.y, sel);
  if (NT == 2) w3_selectors(ch.w1.z, ch.w1.w, ch.w2.x, sel);
  if (NT == 3) w3_selectors(ch.w2.y, ch.w2.z, ch.w2.w, sel);
}
template <int NT>
__device__ __forceinline__ void chunk_selectors(const Chunk2& ch, uint32_t sel[8]) {
  if (NT == 0) w2_selectors(ch.w0.x, ch.w0.y, sel);
  if (NT == 1) w2_selectors(ch.w0.z, ch.w0.w, sel);
  if (NT == 2) w2_selectors(ch.w1.x, ch.w1.y, sel);
  if (NT == 3) w2_selectors(ch.w1.z, ch.w1.w, sel);
}
template <int NT, class C>
__device__ __forceinline__ uint32_t chunk_scales(const C& ch) {
  return NT == 0 ? ch.sc.x : NT == 1 ? ch.sc.y : NT == 2 ? ch.sc.z : ch.sc.w;
}

struct Rows {  // the activation side: four MFMA A fragments (one per 32-group), read from L2
  u32x4_t a0, a1, a2, a3;
};

__device__ __forceinline__ void load_rows(Rows& ch, const uint16_t* arow) {
  ch.a0 = *reinterpret_cast<const u32x4_t*>(arow);
  ch.a1 = *reinterpret_cast<const u32x4_t*>(arow + 32);
  ch.a2 = *reinterpret_cast<const u32x4_t*>(arow + 64);
  ch.a3 = *reinterpret_cast<const u32x4_t*>(arow + 96);
}

__device__ __forceinline__ bf16x8_t expand8(uint32_t sel_lo, uint32_t sel_hi, uint32_t lut_lo, uint32_t lut_hi) {
  const uint32_t f0 = __builtin_amdgcn_perm(lut_hi, lut_lo, sel_lo);
  const uint32_t f1 = __builtin_amdgcn_perm(lut_hi, lut_lo, sel_hi);
  u32x4_t packed;
  packed.x = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(f0, 1.0f, false));
  packed.y = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(f0, 1.0f, true));
  packed.z = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(f1, 1.0f, false));
  packed.w = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(f1, 1.0f, true));
  return __builtin_bit_cast(bf16x8_t, packed);
}

// Half of a 16-row tile of a chunk, sixteen activation rows: 32-groups 0 and 1 (HALF 0: their selectors come from the
// tile's first two code dwords) or 2 and 3 (HALF 1). One MFMA is one group, so the group's scale is folded into the FP32
// accumulator after it, in group order.
template <int HALF, int NT, class C>
__device__ __forceinline__ void compute_half_tile(const C& ch, const u32x4_t& a_lo, const u32x4_t& a_hi, f32x4_t& acc, uint32_t lut_lo, uint32_t lut_hi) {
  const uint32_t scales = chunk_scales<NT>(ch);
  uint32_t sel[8];
  chunk_selectors<NT>(ch, sel);  // the four the half does not use fold away
  const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
  const f32x4_t p0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a_lo), expand8(sel[4 * HALF], sel[4 * HALF + 1], lut_lo, lut_hi), zero, 0, 0, 0);
  const f32x4_t p1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a_hi), expand8(sel[4 * HALF + 2], sel[4 * HALF + 3], lut_lo, lut_hi), zero, 0, 0, 0);
  const float s0 = HALF ? __builtin_amdgcn_cvt_f32_fp8(scales, 2) : __builtin_amdgcn_cvt_f32_fp8(scales, 0);
  const float s1 = HALF ? __builtin_amdgcn_cvt_f32_fp8(scales, 3) : __builtin_amdgcn_cvt_f32_fp8(scales, 1);
  acc.x = fmaf(p1.x, s1, fmaf(p0.x, s0, acc.x));
  acc.y = fmaf(p1.y, s1, fmaf(p0.y, s0, acc.y));
  acc.z = fmaf(p1.z, s1, fmaf(p0.z, s0, acc.z));
  acc.w = fmaf(p1.w, s1, fmaf(p0.w, s0, acc.w));
}

// The four tiles of a chunk over one half of its groups: once a half is done its two activation fragments are free for
// the next chunk's.
template <int HALF, class C>
__device__ __forceinline__ void compute_half_chunk(const C& ch, const u32x4_t& a_lo, const u32x4_t& a_hi, f32x4_t& acc0, f32x4_t& acc1,
                                                   f32x4_t& acc2, f32x4_t& acc3, uint32_t lut_lo, uint32_t lut_hi) {
  compute_half_tile<HALF, 0>(ch, a_lo, a_hi, acc0, lut_lo, lut_hi);
  compute_half_tile<HALF, 1>(ch, a_lo, a_hi, acc1, lut_lo, lut_hi);
  compute_half_tile<HALF, 2>(ch, a_lo, a_hi, acc2, lut_lo, lut_hi);
  compute_half_tile<HALF, 3>(ch, a_lo, a_hi, acc3, lut_lo, lut_hi);
}

// ------------------------------------------------------------------------------------------------ the weight ring
// (ring.hpp) for W3 blocks: three 16-byte loads a lane of codes, one 4-byte load a lane of scales.
// AUX: the loads' cache policy - 2 (non-temporal) for a call that streams far more than the caches hold, 0 for one
// token's few megabytes, which come in faster as ordinary loads.
template <int AUX, int BITS = 3>
struct W3RingOf;

template <int AUX>
struct W3RingOf<AUX, 3> {
  typedef hb::Chunk Chunk;
  static constexpr int BLOCK_BYTES = W3_BLOCK_BYTES, LOADS = 4;
  // the lane's byte offsets in a block for the 16-byte and the 4-byte loads, and where it reads them back
  static __device__ __forceinline__ void lanes(RingSource& src, int lane, int r16, uint32_t slot0, uint32_t& codes, uint32_t& scales) {
    src.codes = 16u * lane;
    src.scales = 4u * lane;
    codes = slot0 + 16u * lane;
    scales = slot0 + 16u * r16;
  }
  static __device__ __forceinline__ void request(const RingSource& src, int chunk, lds_ptr_t slot) {
    const uint32_t at = (uint32_t)chunk * W3_BLOCK_BYTES;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(src.row, slot, 16, src.codes, at, 0, AUX);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(src.row, slot, 16, src.codes, at, 1024, AUX);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(src.row, slot, 16, src.codes, at, 2048, AUX);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(src.row, slot, 4, src.scales, at, W3_SCALE_OFFSET, AUX);
    __builtin_amdgcn_sched_barrier(0);  // asked for here, not wherever the scheduler would sink it below the arithmetic
  }
  // the reads of a block from slot 0, and (after a wait) their values
  static __device__ __forceinline__ void ask(Chunk& ch, uint32_t codes, uint32_t scales) {
    ask_lds<0>(ch.w0, codes);
    ask_lds<1024>(ch.w1, codes);
    ask_lds<2048>(ch.w2, codes);
    ask_lds<W3_SCALE_OFFSET>(ch.sc, scales);
  }
  static __device__ __forceinline__ void have(Chunk& ch) {
    pin(ch.w0);
    pin(ch.w1);
    pin(ch.w2);
    pin(ch.sc);
  }
  template <int BEHIND, int SLOT>  // BEHIND: requests that may stay outstanding
  static __device__ __forceinline__ void take(Chunk& ch, uint32_t codes, uint32_t scales) {
    asm volatile(
        "s_waitcnt vmcnt(%6)\n\t"
        "ds_read_b128 %0, %4 offset:%7\n\t"
        "ds_read_b128 %1, %4 offset:%8\n\t"
        "ds_read_b128 %2, %4 offset:%9\n\t"
        "ds_read_b128 %3, %5 offset:%10\n\t"
        "s_waitcnt lgkmcnt(0)"  // the slot is read: it may be given to another chunk
        : "=&v"(ch.w0), "=&v"(ch.w1), "=&v"(ch.w2), "=&v"(ch.sc)
        : "v"(codes), "v"(scales), "n"(BEHIND), "n"(SLOT * W3_BLOCK_BYTES), "n"(SLOT * W3_BLOCK_BYTES + 1024), "n"(SLOT * W3_BLOCK_BYTES + 2048),
          "n"(SLOT * W3_BLOCK_BYTES + W3_SCALE_OFFSET)
        : "memory");
  }
};
// Two-bit blocks: two 16-byte loads a lane of codes, one 4-byte load a lane of scales; the two slots lie in the same
// LDS a wavefront as a three-bit ring's (the launches size it for either).
template <int AUX>
struct W3RingOf<AUX, 2> {
  typedef hb::Chunk2 Chunk;
  static constexpr int BLOCK_BYTES = W2_BLOCK_BYTES, LOADS = 3;
  static __device__ __forceinline__ void lanes(RingSource& src, int lane, int r16, uint32_t slot0, uint32_t& codes, uint32_t& scales) {
    src.codes = 16u * lane;
    src.scales = 4u * lane;
    codes = slot0 + 16u * lane;
    scales = slot0 + 16u * r16;
  }
  static __device__ __forceinline__ void request(const RingSource& src, int chunk, lds_ptr_t slot) {
    const uint32_t at = (uint32_t)chunk * W2_BLOCK_BYTES;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(src.row, slot, 16, src.codes, at, 0, AUX);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(src.row, slot, 16, src.codes, at, 1024, AUX);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(src.row, slot, 4, src.scales, at, W2_SCALE_OFFSET, AUX);
    __builtin_amdgcn_sched_barrier(0);
  }
  static __device__ __forceinline__ void ask(Chunk& ch, uint32_t codes, uint32_t scales) {
    ask_lds<0>(ch.w0, codes);
    ask_lds<1024>(ch.w1, codes);
    ask_lds<W2_SCALE_OFFSET>(ch.sc, scales);
  }
  static __device__ __forceinline__ void have(Chunk& ch) {
    pin(ch.w0);
    pin(ch.w1);
    pin(ch.sc);
  }
  template <int BEHIND, int SLOT>
  static __device__ __forceinline__ void take(Chunk& ch, uint32_t codes, uint32_t scales) {
    asm volatile(
        "s_waitcnt vmcnt(%5)\n\t"
        "ds_read_b128 %0, %3 offset:%6\n\t"
        "ds_read_b128 %1, %3 offset:%7\n\t"
        "ds_read_b128 %2, %4 offset:%8\n\t"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(ch.w0), "=&v"(ch.w1), "=&v"(ch.sc)
        : "v"(codes), "v"(scales), "n"(BEHIND), "n"(SLOT * W2_BLOCK_BYTES), "n"(SLOT * W2_BLOCK_BYTES + 1024), "n"(SLOT * W2_BLOCK_BYTES + W2_SCALE_OFFSET)
        : "memory");
  }
};
typedef W3RingOf<2> W3Ring;
typedef W3RingOf<0> W3RingCached;
typedef W3RingOf<2, 2> W2Ring;

// A ring that brings in only what the 16-row tiles T0 .. T1 - 1 of a three-bit block need: tile t's three code dwords are
// dwords 3 t .. 3 t + 2 of the lane's twelve, four to a 16-byte load, so the tiles' loads are 3 T0 / 4 .. (3 T1 - 1) / 4 (one
// or two of the three for one tile or a pair of them), and the scales. The Chunk's other registers stay unset and unread.
template <int AUX, int T0, int T1>
struct W3RingPart {
  typedef hb::Chunk Chunk;
  static constexpr int L0 = 3 * T0 / 4, L1 = (3 * T1 - 1) / 4, CODE_LOADS = L1 - L0 + 1;
  static constexpr int BLOCK_BYTES = W3_BLOCK_BYTES, LOADS = CODE_LOADS + 1;
  static_assert(0 <= T0 && T0 < T1 && T1 <= 4 && CODE_LOADS >= 1 && CODE_LOADS <= 2, "a tile or a pair of tiles (the whole block: W3RingOf)");
  static __device__ __forceinline__ void lanes(RingSource& src, int lane, int r16, uint32_t slot0, uint32_t& codes, uint32_t& scales) {
    W3RingOf<AUX>::lanes(src, lane, r16, slot0, codes, scales);
  }
  static __device__ __forceinline__ void request(const RingSource& src, int chunk, lds_ptr_t slot) {
    const uint32_t at = (uint32_t)chunk * W3_BLOCK_BYTES;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(src.row, slot, 16, src.codes, at, 1024 * L0, AUX);
    if (CODE_LOADS == 2) __builtin_amdgcn_raw_ptr_buffer_load_lds(src.row, slot, 16, src.codes, at, 1024 * L1, AUX);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(src.row, slot, 4, src.scales, at, W3_SCALE_OFFSET, AUX);
    __builtin_amdgcn_sched_barrier(0);
  }
  static __device__ __forceinline__ u32x4_t& load_of(Chunk& ch, int l) { return l == 0 ? ch.w0 : l == 1 ? ch.w1 : ch.w2; }
  template <int BEHIND, int SLOT>
  static __device__ __forceinline__ void take(Chunk& ch, uint32_t codes, uint32_t scales) {
    if (CODE_LOADS == 2) {
      asm volatile(
          "s_waitcnt vmcnt(%5)\n\t"
          "ds_read_b128 %0, %3 offset:%6\n\t"
          "ds_read_b128 %1, %3 offset:%7\n\t"
          "ds_read_b128 %2, %4 offset:%8\n\t"
          "s_waitcnt lgkmcnt(0)"
          : "=&v"(load_of(ch, L0)), "=&v"(load_of(ch, L1)), "=&v"(ch.sc)
          : "v"(codes), "v"(scales), "n"(BEHIND), "n"(SLOT * W3_BLOCK_BYTES + 1024 * L0), "n"(SLOT * W3_BLOCK_BYTES + 1024 * L1),
            "n"(SLOT * W3_BLOCK_BYTES + W3_SCALE_OFFSET)
          : "memory");
    } else {
      asm volatile(
          "s_waitcnt vmcnt(%4)\n\t"
          "ds_read_b128 %0, %2 offset:%5\n\t"
          "ds_read_b128 %1, %3 offset:%6\n\t"
          "s_waitcnt lgkmcnt(0)"
          : "=&v"(load_of(ch, L0)), "=&v"(ch.sc)
          : "v"(codes), "v"(scales), "n"(BEHIND), "n"(SLOT * W3_BLOCK_BYTES + 1024 * L0), "n"(SLOT * W3_BLOCK_BYTES + W3_SCALE_OFFSET)
          : "memory");
    }
  }
};
constexpr int RING_BYTES = ring_bytes<W3Ring>();  // LDS per wavefront; its first 4 KB double as the K-split exchange

// ------------------------------------------------------------------------------------------- slots of one to four rows
//
// Most slots of a decode or verify step hold a handful of rows (an expert a few tokens chose). Twelve of the sixteen
// MFMA output rows are then idle, and they can carry the four 32-groups of a chunk instead: A row 4 j + i holds row i of
// the slot over group j's k range only (zero elsewhere), so the four MFMAs of a tile, one per group, chain into ONE
// accumulator whose rows 4 j .. 4 j + 3 are group j's partial sums. Lane (q, r16) then holds group q's sums for the
// slot's four rows: one scale conversion and four multiply-adds per tile instead of four and sixteen, and sixteen bytes
// of activations per lane and chunk instead of sixty-four. The four groups are added once, after the last chunk, in the
// exchange through LDS that the K splits are added in.
constexpr int FEW_ROWS = 4;

// fc2 stores by pair index, which it reads from the sorted list: asked for ahead of the weights, so that the epilogue
// does not wait on memory once more.
struct FewPairs {
  int pair[FEW_ROWS];
  __device__ __forceinline__ void ask(const StreamParams& p, const Slot& sl, int row0) {
#pragma unroll
    for (int r = 0; r < FEW_ROWS; r++) pair[r] = p.order[sl.p0 + min(row0 + r, sl.rows - 1)];
  }
  __device__ __forceinline__ int of(int r) const { return r == 0 ? pair[0] : r == 1 ? pair[1] : r == 2 ? pair[2] : pair[3]; }
};

__device__ __forceinline__ void store_pair(const StreamParams& p, int64_t pair, int n, float y) {
  if (p.out_bf16) {
    reinterpret_cast<uint16_t*>(p.out)[pair * p.out_stride + n] = bf16_of(y);
  } else {
    reinterpret_cast<float*>(p.out)[pair * p.out_stride + n] = y;
  }
}

template <int NT, class C>
__device__ __forceinline__ void compute_tile_few(const C& w, const Rows& ch, f32x4_t& acc, uint32_t lut_lo, uint32_t lut_hi, uint32_t q8) {
  const uint32_t scales = chunk_scales<NT>(w);
  uint32_t sel[8];
  chunk_selectors<NT>(w, sel);
  f32x4_t part = {0.f, 0.f, 0.f, 0.f};
  part = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, ch.a0), expand8(sel[0], sel[1], lut_lo, lut_hi), part, 0, 0, 0);
  part = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, ch.a1), expand8(sel[2], sel[3], lut_lo, lut_hi), part, 0, 0, 0);
  part = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, ch.a2), expand8(sel[4], sel[5], lut_lo, lut_hi), part, 0, 0, 0);
  part = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, ch.a3), expand8(sel[6], sel[7], lut_lo, lut_hi), part, 0, 0, 0);
  const float s = __builtin_amdgcn_cvt_f32_fp8(scales >> q8, 0);  // the scale of this lane's group
  acc.x = fmaf(part.x, s, acc.x);
  acc.y = fmaf(part.y, s, acc.y);
  acc.z = fmaf(part.z, s, acc.z);
  acc.w = fmaf(part.w, s, acc.w);
}

// The E4M3-activation form of the four-row body (the arithmetic of the reference kernel, hibana/kernels/csrc/
// w3_gemm.cu:105-108: FP8 x FP8 products, FP32 sums a group, the two group scales folded into the accumulator). The
// codebook's E4M3 bytes are the MFMA operand as they come out of v_perm_b32: no conversion. `a`: the lane's eight
// activation codes of the chunk; xs: the activation scales of the slot's four rows at this lane's group.
__device__ __forceinline__ long fp8x8(uint32_t lo, uint32_t hi) { return (long)(((uint64_t)hi << 32) | lo); }

template <int NT, class C>
__device__ __forceinline__ void compute_tile_few8(const C& w, const long a[4], const f32x4_t& xs, f32x4_t& acc, uint32_t lut_lo, uint32_t lut_hi,
                                                  uint32_t q8) {
  const uint32_t scales = chunk_scales<NT>(w);
  uint32_t sel[8];
  chunk_selectors<NT>(w, sel);
  f32x4_t part = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int j = 0; j < 4; j++) {
    const long b = fp8x8(__builtin_amdgcn_perm(lut_hi, lut_lo, sel[2 * j]), __builtin_amdgcn_perm(lut_hi, lut_lo, sel[2 * j + 1]));
    part = __builtin_amdgcn_mfma_f32_16x16x32_fp8_fp8(a[j], b, part, 0, 0, 0);
  }
  const float s = __builtin_amdgcn_cvt_f32_fp8(scales >> q8, 0);  // the weight scale of this lane's group
  acc.x = fmaf(part.x, xs.x * s, acc.x);
  acc.y = fmaf(part.y, xs.y * s, acc.y);
  acc.z = fmaf(part.z, xs.z * s, acc.z);
  acc.w = fmaf(part.w, xs.w * s, acc.w);
}

template <int T0 = 0, int T1 = 4, class C>  // the 16-row tiles T0 .. T1 - 1 of the block
__device__ __forceinline__ void compute_few8(const C& ch, long a, const f32x4_t& xs, int grp, f32x4_t& acc0, f32x4_t& acc1, f32x4_t& acc2,
                                             f32x4_t& acc3, uint32_t lut_lo, uint32_t lut_hi, uint32_t q8) {
  long rows[4];  // MFMA j's A operand: the lane's codes in its own group, zero in the others
#pragma unroll
  for (int j = 0; j < 4; j++) rows[j] = grp == j ? a : 0L;
  if (T0 <= 0 && 0 < T1) compute_tile_few8<0>(ch, rows, xs, acc0, lut_lo, lut_hi, q8);
  if (T0 <= 1 && 1 < T1) compute_tile_few8<1>(ch, rows, xs, acc1, lut_lo, lut_hi, q8);
  if (T0 <= 2 && 2 < T1) compute_tile_few8<2>(ch, rows, xs, acc2, lut_lo, lut_hi, q8);
  if (T0 <= 3 && 3 < T1) compute_tile_few8<3>(ch, rows, xs, acc3, lut_lo, lut_hi, q8);
}

// `a`: the lane's sixteen activation bytes of the chunk (row r16 % 4 of the slot, the k range of group r16 / 4 that this
// lane owns in the MFMA A operand); grp: that group.
template <class C>
__device__ __forceinline__ void compute_few(const C& ch, const u32x4_t& a, int grp, f32x4_t& acc0, f32x4_t& acc1, f32x4_t& acc2,
                                            f32x4_t& acc3, uint32_t lut_lo, uint32_t lut_hi, uint32_t q8) {
  const u32x4_t none = {0u, 0u, 0u, 0u};
  Rows rows;  // MFMA j's A operand: the lane's bytes in its own group, zero in the others
  rows.a0 = grp == 0 ? a : none;
  rows.a1 = grp == 1 ? a : none;
  rows.a2 = grp == 2 ? a : none;
  rows.a3 = grp == 3 ? a : none;
  compute_tile_few<0>(ch, rows, acc0, lut_lo, lut_hi, q8);
  compute_tile_few<1>(ch, rows, acc1, lut_lo, lut_hi, q8);
  compute_tile_few<2>(ch, rows, acc2, lut_lo, lut_hi, q8);
  compute_tile_few<3>(ch, rows, acc3, lut_lo, lut_hi, q8);
}

// The two bodies of the stream differ in the activations: what registers they keep, when they ask for them, how a
// chunk is computed. `step<ODD, MORE2, MORE1>` computes chunk i (ODD: its parity; MORE2 / MORE1: chunks i + 2 / i + 1
// exist) and asks for the activations whose registers it frees.
struct FewActs {
  static constexpr int LOADS = 1;  // activation loads per chunk
  u32x4_t held[2];                 // the lane's sixteen bytes of the next even and the next odd chunk
  int grp;
  uint32_t q8;
  const uint16_t* at;              // the lane's sixteen bytes of the wavefront's first chunk
  __device__ __forceinline__ u32x4_t load(int i) const { return *reinterpret_cast<const u32x4_t*>(at + (int64_t)i * 128); }
  template <int EPI>
  __device__ __forceinline__ void start(const StreamParams& p, const Slot& sl, int row0, int c0, int n, int lane) {
    const int q = lane >> 4, r16 = lane & 15;
    grp = r16 >> 2;
    at = activation_row<EPI>(p, sl, row0 + (r16 & 3)) + (int64_t)c0 * 128 + 32 * grp + 8 * q;
    q8 = 8 * q;
    held[0] = load(0);
    if (n > 1) held[1] = load(1);
  }
  template <int ODD, bool MORE2, bool MORE1, class C>
  __device__ __forceinline__ void step(const C& ch, int i, f32x4_t& acc0, f32x4_t& acc1, f32x4_t& acc2, f32x4_t& acc3, const Slot& sl) {
    compute_few(ch, held[ODD], grp, acc0, acc1, acc2, acc3, sl.lut_lo, sl.lut_hi, q8);
    if (MORE2) held[ODD] = load(i + 2);
  }
};

// FewActs over the 16-row tiles T0 .. T1 - 1 of the block only (the other accumulators stay zero).
template <int T0, int T1>
struct FewActsPart : FewActs {
  template <int ODD, bool MORE2, bool MORE1, class C>
  __device__ __forceinline__ void step(const C& ch, int i, f32x4_t& acc0, f32x4_t& acc1, f32x4_t& acc2, f32x4_t& acc3, const Slot& sl) {
    const u32x4_t none = {0u, 0u, 0u, 0u};
    const u32x4_t a = held[ODD];
    Rows rows;  // as compute_few: the lane's bytes in its own group, zero in the others
    rows.a0 = grp == 0 ? a : none;
    rows.a1 = grp == 1 ? a : none;
    rows.a2 = grp == 2 ? a : none;
    rows.a3 = grp == 3 ? a : none;
    if (T0 <= 0 && 0 < T1) compute_tile_few<0>(ch, rows, acc0, sl.lut_lo, sl.lut_hi, q8);
    if (T0 <= 1 && 1 < T1) compute_tile_few<1>(ch, rows, acc1, sl.lut_lo, sl.lut_hi, q8);
    if (T0 <= 2 && 2 < T1) compute_tile_few<2>(ch, rows, acc2, sl.lut_lo, sl.lut_hi, q8);
    if (T0 <= 3 && 3 < T1) compute_tile_few<3>(ch, rows, acc3, sl.lut_lo, sl.lut_hi, q8);
    if (MORE2) held[ODD] = load(i + 2);
  }
};

struct FewActs8 {  // E4M3 activations: eight codes a lane and chunk, and the scales of the slot's four rows at the lane's output group
  static constexpr int LOADS = 5;
  long held[2];
  f32x4_t scale[2];
  int grp;
  uint32_t q8;
  const uint8_t* at;       // the lane's eight codes of the wavefront's first chunk
  const float* scales;     // the scale matrix
  uint32_t soff[4];        // in it, the scale of slot row row0 + i at group q of that chunk (the launch keeps the matrix under 2^32 scales)
  __device__ __forceinline__ void load(int slot, int i) {
    held[slot] = *reinterpret_cast<const long*>(at + (int64_t)i * 128);
    scale[slot] = f32x4_t{scales[soff[0] + 4 * i], scales[soff[1] + 4 * i], scales[soff[2] + 4 * i], scales[soff[3] + 4 * i]};
  }
  template <int EPI>
  __device__ __forceinline__ void start(const StreamParams& p, const Slot& sl, int row0, int c0, int n, int lane) {
    const int q = lane >> 4, r16 = lane & 15;
    grp = r16 >> 2;
    at = p.aq + activation_row_index<EPI>(p, sl, row0 + (r16 & 3)) * p.a_stride + (int64_t)c0 * 128 + 32 * grp + 8 * q;
    scales = p.aq_scale;
#pragma unroll
    for (int i = 0; i < 4; i++) soff[i] = (uint32_t)(activation_row_index<EPI>(p, sl, row0 + i) * (p.a_stride >> 5)) + 4 * c0 + q;
    q8 = 8 * q;
    load(0, 0);
    if (n > 1) load(1, 1);
  }
  template <int ODD, bool MORE2, bool MORE1, class C>
  __device__ __forceinline__ void step(const C& ch, int i, f32x4_t& acc0, f32x4_t& acc1, f32x4_t& acc2, f32x4_t& acc3, const Slot& sl) {
    compute_few8(ch, held[ODD], scale[ODD], grp, acc0, acc1, acc2, acc3, sl.lut_lo, sl.lut_hi, q8);
    if (MORE2) load(ODD, i + 2);
  }
};

// FewActs8 over the 16-row tiles T0 .. T1 - 1 of the block only (the other accumulators stay zero).
template <int T0, int T1>
struct FewActs8Part : FewActs8 {
  template <int ODD, bool MORE2, bool MORE1, class C>
  __device__ __forceinline__ void step(const C& ch, int i, f32x4_t& acc0, f32x4_t& acc1, f32x4_t& acc2, f32x4_t& acc3, const Slot& sl) {
    compute_few8<T0, T1>(ch, held[ODD], scale[ODD], grp, acc0, acc1, acc2, acc3, sl.lut_lo, sl.lut_hi, q8);
    if (MORE2) load(ODD, i + 2);
  }
};

// Slots of at most TWO rows on the two-plane form of the activations (split_row: x = (hi + lo) * s, both E4M3), on
// v_mfma_f32_16x16x32_fp8_fp8: both planes of both rows ride in the four A rows of a group - A row 4 g + 2 plane + t is
// plane `plane` of slot row t over group g only - so the MFMA count is the BF16 body's (one a group and tile), the
// weights are the codebook's E4M3 bytes as v_perm_b32 delivers them (no conversion: 132 VALU instructions a chunk
// instead of 204) and an A operand is two registers. Both planes are in the same units and their sums add in
// finish_few, where the row's activation scale multiplies the result. Register i of lane (q, r16) of a tile's result is group q's sum for
// plane i / 2 of slot row i % 2 and weight row r16; finish_few adds the planes.
struct FewPlaneActs {
  static constexpr int LOADS = 1;
  long held[2];       // the lane's eight E4M3 bytes (its row, plane and group) of the next even and the next odd chunk
  int grp;
  uint32_t q8;
  const uint8_t* at;  // ... of the wavefront's first chunk
  __device__ __forceinline__ long load(int i) const { return *reinterpret_cast<const long*>(at + (int64_t)i * 256); }
  template <int EPI>
  __device__ __forceinline__ void start(const StreamParams& p, const Slot& sl, int row0, int c0, int n, int lane) {
    const int q = lane >> 4, r16 = lane & 15;
    grp = r16 >> 2;
    q8 = 8 * q;
    at = p.a2 + activation_row_index<EPI>(p, sl, row0 + (r16 & 1)) * (2 * p.a_stride) + (int64_t)c0 * 256 + 64 * (r16 & 2) + 32 * grp + 8 * q;
    held[0] = load(0);
    if (n > 1) held[1] = load(1);
  }
  template <int NT, class C>
  static __device__ __forceinline__ void tile(const C& w, const long a[4], f32x4_t& acc, uint32_t lut_lo, uint32_t lut_hi, uint32_t q8) {
    const uint32_t scales = chunk_scales<NT>(w);
    uint32_t sel[8];
    chunk_selectors<NT>(w, sel);
    f32x4_t part = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const long b = fp8x8(__builtin_amdgcn_perm(lut_hi, lut_lo, sel[2 * j]), __builtin_amdgcn_perm(lut_hi, lut_lo, sel[2 * j + 1]));
      part = __builtin_amdgcn_mfma_f32_16x16x32_fp8_fp8(a[j], b, part, 0, 0, 0);
    }
    const float s = __builtin_amdgcn_cvt_f32_fp8(scales >> q8, 0);  // the scale of this lane's group
    acc.x = fmaf(part.x, s, acc.x);
    acc.y = fmaf(part.y, s, acc.y);
    acc.z = fmaf(part.z, s, acc.z);
    acc.w = fmaf(part.w, s, acc.w);
  }
  template <int ODD, bool MORE2, bool MORE1, class C>
  __device__ __forceinline__ void step(const C& ch, int i, f32x4_t& acc0, f32x4_t& acc1, f32x4_t& acc2, f32x4_t& acc3, const Slot& sl) {
    long rows[4];  // MFMA j's A operand: the lane's bytes in its own group, zero in the others
#pragma unroll
    for (int j = 0; j < 4; j++) rows[j] = grp == j ? held[ODD] : 0L;
    tile<0>(ch, rows, acc0, sl.lut_lo, sl.lut_hi, q8);
    tile<1>(ch, rows, acc1, sl.lut_lo, sl.lut_hi, q8);
    tile<2>(ch, rows, acc2, sl.lut_lo, sl.lut_hi, q8);
    tile<3>(ch, rows, acc3, sl.lut_lo, sl.lut_hi, q8);
    if (MORE2) held[ODD] = load(i + 2);
  }
};
constexpr int PLANE_ROWS = 2;

// The activation scales of a slot's (up to) four rows, asked for ahead of the weights like the pair indices.
struct FewScales {
  float s[FEW_ROWS];
  template <int EPI>
  __device__ __forceinline__ void ask(const StreamParams& p, const Slot& sl, int row0) {
#pragma unroll
    for (int r = 0; r < FEW_ROWS; r++) s[r] = p.a2_scale[activation_row_index<EPI>(p, sl, row0 + r)];
  }
  __device__ __forceinline__ float of(int r) const { return r == 0 ? s[0] : r == 1 ? s[1] : r == 2 ? s[2] : s[3]; }
};

struct FullActs {  // up to sixteen rows: lane (q, r16) feeds row r16, k 8 q .. 8 q + 7 of every group
  static constexpr int LOADS = 4;
  Rows held;           // one chunk's fragments; each half is asked for again as soon as its groups are done
  const uint16_t* at;
  template <int EPI>
  __device__ __forceinline__ void start(const StreamParams& p, const Slot& sl, int, int c0, int, int lane) {
    at = activation_row<EPI>(p, sl, lane & 15) + (int64_t)c0 * 128 + 8 * (lane >> 4);
    load_rows(held, at);
  }
  template <int ODD, bool MORE2, bool MORE1, class C>
  __device__ __forceinline__ void step(const C& ch, int i, f32x4_t& acc0, f32x4_t& acc1, f32x4_t& acc2, f32x4_t& acc3, const Slot& sl) {
    const uint16_t* next = at + (int64_t)(i + 1) * 128;
    compute_half_chunk<0>(ch, held.a0, held.a1, acc0, acc1, acc2, acc3, sl.lut_lo, sl.lut_hi);
    if (MORE1) {
      held.a0 = *reinterpret_cast<const u32x4_t*>(next);
      held.a1 = *reinterpret_cast<const u32x4_t*>(next + 32);
    }
    compute_half_chunk<1>(ch, held.a2, held.a3, acc0, acc1, acc2, acc3, sl.lut_lo, sl.lut_hi);
    if (MORE1) {
      held.a2 = *reinterpret_cast<const u32x4_t*>(next + 64);
      held.a3 = *reinterpret_cast<const u32x4_t*>(next + 96);
    }
  }
};

// The same of a routed slot, with two chunks' activations held and a chunk's asked for two chunks ahead, as its block is: asked for one chunk ahead
// they stand behind a block asked for one chunk ago, and in a launch of few wavefronts a unit every chunk waits for memory: 40 rows
// under a budget of 64 experts (2048, 512) 50.7 us, so 50.0. Dense calls, whose wavefronts have few chunks, lose by the second chunk's loads ahead of
// the first product: 8192 x 2048 twelve rows 6.2 us, so 6.5; 51200 x 2048 17.3 and 16.7.
struct FullActsAhead {
  static constexpr int LOADS = 4;
  Rows even, odd;
  const uint16_t* at;
  template <int EPI>
  __device__ __forceinline__ void start(const StreamParams& p, const Slot& sl, int, int c0, int n, int lane) {
    at = activation_row<EPI>(p, sl, lane & 15) + (int64_t)c0 * 128 + 8 * (lane >> 4);
    load_rows(even, at);
    if (n > 1) load_rows(odd, at + 128);
  }
  template <int ODD, bool MORE2, bool MORE1, class C>
  __device__ __forceinline__ void step(const C& ch, int i, f32x4_t& acc0, f32x4_t& acc1, f32x4_t& acc2, f32x4_t& acc3, const Slot& sl) {
    Rows& held = ODD ? odd : even;
    compute_half_chunk<0>(ch, held.a0, held.a1, acc0, acc1, acc2, acc3, sl.lut_lo, sl.lut_hi);
    compute_half_chunk<1>(ch, held.a2, held.a3, acc0, acc1, acc2, acc3, sl.lut_lo, sl.lut_hi);
    if (MORE2) load_rows(held, at + (int64_t)(i + 2) * 128);
  }
};

// The sixteen-row body on E4M3 activations: lane (q, r16) feeds row r16's eight codes of every group (the FP8 MFMA's A
// operand) and folds, per group, the product of the weight scale and the activation scales of the four rows its
// accumulator registers hold (rows 4 q .. 4 q + 3). Both are asked for again by halves, as FullActs does.
struct FullActs8 {
  typedef __attribute__((ext_vector_type(2))) float f32x2_t;
  static constexpr int LOADS = 8;  // four of codes and at least four of scales: of a row's two scale pairs, asked for side by side, the compiler makes one load
  long a[4];            // the lane's codes of groups 0..3
  f32x2_t xs_lo[4];     // activation scales of rows 4 q + r at groups 0, 1
  f32x2_t xs_hi[4];     // ... at groups 2, 3
  const uint8_t* at;    // the lane's codes of group 0 of the wavefront's first chunk
  const float* scales;
  uint32_t soff[4];     // the scale of slot row 4 q + r at group 0 of that chunk
  __device__ __forceinline__ void load_half(int half, int i) {
    a[2 * half] = *reinterpret_cast<const long*>(at + (int64_t)i * 128 + 64 * half);
    a[2 * half + 1] = *reinterpret_cast<const long*>(at + (int64_t)i * 128 + 64 * half + 32);
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const f32x2_t v = *reinterpret_cast<const f32x2_t*>(scales + soff[r] + 4 * i + 2 * half);
      if (half) {
        xs_hi[r] = v;
      } else {
        xs_lo[r] = v;
      }
    }
  }
  template <int EPI>
  __device__ __forceinline__ void start(const StreamParams& p, const Slot& sl, int, int c0, int, int lane) {
    const int q = lane >> 4, r16 = lane & 15;
    at = p.aq + activation_row_index<EPI>(p, sl, r16) * p.a_stride + (int64_t)c0 * 128 + 8 * q;
    scales = p.aq_scale;
#pragma unroll
    for (int r = 0; r < 4; r++) soff[r] = (uint32_t)(activation_row_index<EPI>(p, sl, 4 * q + r) * (p.a_stride >> 5)) + 4 * c0;
    load_half(0, 0);
    load_half(1, 0);
  }
  // groups 2 HALF and 2 HALF + 1 of tile NT
  template <int HALF, int NT, class C>
  __device__ __forceinline__ void half_tile(const C& ch, f32x4_t& acc, uint32_t lut_lo, uint32_t lut_hi) const {
    const uint32_t sc = chunk_scales<NT>(ch);
    uint32_t sel[8];
    chunk_selectors<NT>(ch, sel);  // the four the half does not use fold away
#pragma unroll
    for (int jj = 0; jj < 2; jj++) {
      const int j = 2 * HALF + jj;
      const long b = fp8x8(__builtin_amdgcn_perm(lut_hi, lut_lo, sel[2 * j]), __builtin_amdgcn_perm(lut_hi, lut_lo, sel[2 * j + 1]));
      const f32x4_t part = __builtin_amdgcn_mfma_f32_16x16x32_fp8_fp8(a[j], b, f32x4_t{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
      const float ws = j == 0 ? __builtin_amdgcn_cvt_f32_fp8(sc, 0) : j == 1 ? __builtin_amdgcn_cvt_f32_fp8(sc, 1)
                     : j == 2 ? __builtin_amdgcn_cvt_f32_fp8(sc, 2) : __builtin_amdgcn_cvt_f32_fp8(sc, 3);
      const f32x2_t* xs = HALF ? xs_hi : xs_lo;
      acc.x = fmaf(part.x, (jj ? xs[0].y : xs[0].x) * ws, acc.x);
      acc.y = fmaf(part.y, (jj ? xs[1].y : xs[1].x) * ws, acc.y);
      acc.z = fmaf(part.z, (jj ? xs[2].y : xs[2].x) * ws, acc.z);
      acc.w = fmaf(part.w, (jj ? xs[3].y : xs[3].x) * ws, acc.w);
    }
  }
  // ... of the four tiles
  template <int HALF, class C>
  __device__ __forceinline__ void half_chunk(const C& ch, f32x4_t& acc0, f32x4_t& acc1, f32x4_t& acc2, f32x4_t& acc3, uint32_t lut_lo,
                                             uint32_t lut_hi) const {
    half_tile<HALF, 0>(ch, acc0, lut_lo, lut_hi);
    half_tile<HALF, 1>(ch, acc1, lut_lo, lut_hi);
    half_tile<HALF, 2>(ch, acc2, lut_lo, lut_hi);
    half_tile<HALF, 3>(ch, acc3, lut_lo, lut_hi);
  }
  template <int ODD, bool MORE2, bool MORE1, class C>
  __device__ __forceinline__ void step(const C& ch, int i, f32x4_t& acc0, f32x4_t& acc1, f32x4_t& acc2, f32x4_t& acc3, const Slot& sl) {
    half_chunk<0>(ch, acc0, acc1, acc2, acc3, sl.lut_lo, sl.lut_hi);
    if (MORE1) load_half(0, i + 1);
    half_chunk<1>(ch, acc0, acc1, acc2, acc3, sl.lut_lo, sl.lut_hi);
    if (MORE1) load_half(1, i + 1);
  }
};

// The sixteen-row bodies over the 16-row tiles T0 .. T1 - 1 of the block only (the other accumulators stay zero).
template <int T0, int T1>
struct FullActsPart : FullActs {
  template <int HALF, class C>
  static __device__ __forceinline__ void half(const C& ch, const u32x4_t& a_lo, const u32x4_t& a_hi, f32x4_t& acc0, f32x4_t& acc1, f32x4_t& acc2, f32x4_t& acc3,
                                              const Slot& sl) {
    if (T0 <= 0 && 0 < T1) compute_half_tile<HALF, 0>(ch, a_lo, a_hi, acc0, sl.lut_lo, sl.lut_hi);
    if (T0 <= 1 && 1 < T1) compute_half_tile<HALF, 1>(ch, a_lo, a_hi, acc1, sl.lut_lo, sl.lut_hi);
    if (T0 <= 2 && 2 < T1) compute_half_tile<HALF, 2>(ch, a_lo, a_hi, acc2, sl.lut_lo, sl.lut_hi);
    if (T0 <= 3 && 3 < T1) compute_half_tile<HALF, 3>(ch, a_lo, a_hi, acc3, sl.lut_lo, sl.lut_hi);
  }
  template <int ODD, bool MORE2, bool MORE1, class C>
  __device__ __forceinline__ void step(const C& ch, int i, f32x4_t& acc0, f32x4_t& acc1, f32x4_t& acc2, f32x4_t& acc3, const Slot& sl) {
    const uint16_t* next = at + (int64_t)(i + 1) * 128;
    half<0>(ch, held.a0, held.a1, acc0, acc1, acc2, acc3, sl);
    if (MORE1) {
      held.a0 = *reinterpret_cast<const u32x4_t*>(next);
      held.a1 = *reinterpret_cast<const u32x4_t*>(next + 32);
    }
    half<1>(ch, held.a2, held.a3, acc0, acc1, acc2, acc3, sl);
    if (MORE1) {
      held.a2 = *reinterpret_cast<const u32x4_t*>(next + 64);
      held.a3 = *reinterpret_cast<const u32x4_t*>(next + 96);
    }
  }
};
template <int T0, int T1>
struct FullActs8Part : FullActs8 {
  template <int HALF, class C>
  __device__ __forceinline__ void half(const C& ch, f32x4_t& acc0, f32x4_t& acc1, f32x4_t& acc2, f32x4_t& acc3, const Slot& sl) const {
    if (T0 <= 0 && 0 < T1) half_tile<HALF, 0>(ch, acc0, sl.lut_lo, sl.lut_hi);
    if (T0 <= 1 && 1 < T1) half_tile<HALF, 1>(ch, acc1, sl.lut_lo, sl.lut_hi);
    if (T0 <= 2 && 2 < T1) half_tile<HALF, 2>(ch, acc2, sl.lut_lo, sl.lut_hi);
    if (T0 <= 3 && 3 < T1) half_tile<HALF, 3>(ch, acc3, sl.lut_lo, sl.lut_hi);
  }
  template <int ODD, bool MORE2, bool MORE1, class C>
  __device__ __forceinline__ void step(const C& ch, int i, f32x4_t& acc0, f32x4_t& acc1, f32x4_t& acc2, f32x4_t& acc3, const Slot& sl) {
    half<0>(ch, acc0, acc1, acc2, acc3, sl);
    if (MORE1) load_half(0, i + 1);
    half<1>(ch, acc0, acc1, acc2, acc3, sl);
    if (MORE1) load_half(1, i + 1);
  }
};

// The end of a 64-row block for a slot of at most four rows. Lane (g, r16) of each of the block's K splits holds, in
// register r of accumulator t, group g's part of (tile t, slot row r, column r16): sixteen values a lane, each to be
// added over the four groups and the splits. They go to LDS, and the workgroup's 64 x ks lanes share the 16 x 16
// results of the block: lane (q, r16) of split `ks` takes tile q, column r16, of slot rows row0 + ks, row0 + ks + p.ks, ... It
// multiplies by its tile's row scale (`scale`, asked for before the first chunk); a gated pair's gate comes from the
// neighbouring tile's lane. Every wavefront of the workgroup must call it when K is split (one workgroup barrier).
// QUANT (fc1 in the E4M3 activation mode): h leaves as codes and scales; a 32-group is two of the wavefront's DPP rows.
template <int EPI, bool QUANT = false, bool SCALED = false, bool PLANES = false>  // SCALED: the sums are of the two-plane activations and take their row's scale; PLANES: registers 2, 3 hold the lower plane of rows 0, 1
__device__ __forceinline__ void finish_few(const StreamParams& p, const Slot& sl, int row0, float scale, int nb, bool active, int wave, int ks,
                                           int nbi, float* partial, const f32x4_t& acc0, const f32x4_t& acc1, const f32x4_t& acc2,
                                           const f32x4_t& acc3, const FewPairs& pairs = FewPairs{}, const FewScales& xs = FewScales{}, int t0 = 0, int t1 = 4) {
  constexpr int STRIDE = RING_BYTES / 4;
  const int lane = threadIdx.x & 63, q = lane >> 4, r16 = lane & 15;
  float* mine = partial + wave * STRIDE;
  const f32x4_t all[4] = {acc0, acc1, acc2, acc3};
#pragma unroll
  for (int t = 0; t < 4; t++) {
    mine[(t * 4 + 0) * 64 + lane] = all[t].x;
    mine[(t * 4 + 1) * 64 + lane] = all[t].y;
    mine[(t * 4 + 2) * 64 + lane] = all[t].z;
    mine[(t * 4 + 3) * 64 + lane] = all[t].w;
  }
  if (p.ks > 1) {
    __syncthreads();
  } else {
    __builtin_amdgcn_wave_barrier();  // the lanes of one wavefront: its LDS operations execute in program order
  }
  if (!active || q < t0 || q >= t1) return;  // (fewer than all four tiles: dense calls, which exchange nothing between lanes below)
  const float* first = partial + nbi * p.ks * STRIDE + r16;
  const int rows = min(PLANES ? PLANE_ROWS : FEW_ROWS, sl.rows - row0);
  for (int r = ks; r < rows; r += p.ks) {
    const float* at = first + (q * 4 + r) * 64;
    float v = 0.f;
    for (int s = 0; s < p.ks; s++) {
      v += (at[0] + at[16]) + (at[32] + at[48]);
      if (PLANES) v += (at[128] + at[144]) + (at[160] + at[176]);
      at += STRIDE;
    }
    const float y = SCALED ? v * scale * xs.of(r) : v * scale;
    if (EPI == EPI_FC1_GATED) {
      const float gate = __shfl_xor(y, 16);  // tiles 2 t and 2 t + 1 are a pair's up and gate rows
      if (QUANT) {  // the pairs are in tiles 0 and 2: their two rows of lanes are the group
        const bool pair = (q & 1) == 0;
        const float h = pair ? fc1_value<EPI>(y, gate) : 0.f;
        float amax = row16_max(fabsf(h));
        amax = fmaxf(amax, __shfl_xor(amax, 32));
        if (pair) store_quantized(p, sl.p0 + row0 + r, nb * 32 + 8 * q + r16, h, amax, lane == 0);
      } else if ((q & 1) == 0) {
        store_out<EPI>(p, sl, nb, q >> 1, row0 + r, r16, y, gate);
      }
    } else if (QUANT) {  // tiles 0, 1 and tiles 2, 3 are the block's two groups
      const float h = fc1_value<EPI>(y, 0.f);
      float amax = row16_max(fabsf(h));
      amax = fmaxf(amax, __shfl_xor(amax, 16));
      store_quantized(p, sl.p0 + row0 + r, nb * 64 + 16 * q + r16, h, amax, (lane & 31) == 0);
    } else if (EPI == EPI_FC2) {
      store_pair(p, pairs.of(r), nb * 64 + lane, y);  // lane (q, r16) is column 16 q + r16 of the block
    } else {
      store_out<EPI>(p, sl, nb, q, row0 + r, r16, y, 0.f);
    }
  }
}

// General kernel, any K: one workgroup per (run of p.nbw 64-row blocks, slot), K split p.ks ways across its wavefronts.
// A8: E4M3 activations (p.aq, p.aq_scale), with the two bodies' FP8 forms; fc1 then writes h as E4M3 codes and
// scales (p.oq, p.oq_scale), the activation rounding done in its epilogue.
// SPLIT: slots of at most two rows read the two-plane form of the activations (p.a2) and run on the FP8 matrix cores.
// One workgroup's work: slot `sl` (with rows), the run `bx` of p.nbw 64-row blocks; `rings`: the launch's dynamic LDS.
template <int EPI, bool A8, bool SPLIT, class Ring = W3Ring, class Wait>
__device__ __forceinline__ void stream_workgroup(const StreamParams& p, const Slot& sl, int bx, uint8_t* rings, Wait& wait) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // the same in every lane: kept in scalars
  const WaveShare share = wave_share(p, wave);
  const int ks = share.ks, nbi = share.nbi, nb = bx * p.nbw + nbi;
  const bool active = nb < p.n_blocks;
  f32x4_t acc0 = {0.f, 0.f, 0.f, 0.f}, acc1 = acc0, acc2 = acc0, acc3 = acc0;
  uint8_t* ring = rings + wave * RING_BYTES;
  if (Wait::WAITS && !active) wait.done();
  constexpr bool QUANT = A8 && epi_gathers(EPI);  // fc1 on E4M3 activations hands fc2 E4M3 activations
  if (A8) {
    if (sl.rows <= FEW_ROWS) {  // uniform over the workgroup
      float scale = 0.f;
      FewPairs pairs{};
      if (active) {
        scale = sl.rs[nb * 64 + lane];
        if (EPI == EPI_FC2) pairs.ask(p, sl, 0);
        stream_block_behind<EPI, FewActs8, Ring>(p, sl, 0, nb, share.c0, share.c1, lane, ring, acc0, acc1, acc2, acc3, wait);
      }
      if (!wait.there) return;
      finish_few<EPI, QUANT>(p, sl, 0, scale, nb, active, wave, ks, nbi, reinterpret_cast<float*>(rings), acc0, acc1, acc2, acc3, pairs);
    } else {
      RowScales rs{};
      if (active) {
        stream_block_behind<EPI, FullActs8, Ring>(p, sl, 0, nb, share.c0, share.c1, lane, ring, acc0, acc1, acc2, acc3, wait);
        rs = row_scales<true>(sl, nb, lane & 15);
      }
      if (!wait.there) return;
      finish_block<EPI, true, RING_BYTES / 4, QUANT>(p, sl, rs, nb, active, ks, nbi, reinterpret_cast<float*>(rings), acc0, acc1, acc2, acc3);
    }
  } else if (SPLIT && sl.rows <= PLANE_ROWS) {  // uniform over the workgroup
    float scale = 0.f;
    FewPairs pairs{};
    FewScales xs{};
    if (active) {
      scale = sl.rs[nb * 64 + lane];
      if (EPI == EPI_FC2) pairs.ask(p, sl, 0);
      xs.ask<EPI>(p, sl, 0);
      stream_block_behind<EPI, FewPlaneActs, Ring>(p, sl, 0, nb, share.c0, share.c1, lane, ring, acc0, acc1, acc2, acc3, wait);
    }
    if (!wait.there) return;
    finish_few<EPI, false, true, true>(p, sl, 0, scale, nb, active, wave, ks, nbi, reinterpret_cast<float*>(rings), acc0, acc1, acc2, acc3, pairs, xs);
  } else if (sl.rows <= FEW_ROWS && !p.no_few) {  // uniform over the workgroup
    float scale = 0.f;
    FewPairs pairs{};
    if (active) {
      scale = sl.rs[nb * 64 + lane];  // row 16 q + r16 of the block: asked for ahead of the chunks, there when the epilogue wants it
      if (EPI == EPI_FC2) pairs.ask(p, sl, 0);
      stream_block_behind<EPI, FewActs, Ring>(p, sl, 0, nb, share.c0, share.c1, lane, ring, acc0, acc1, acc2, acc3, wait);  // at least one chunk: ks <= chunks
    }
    if (!wait.there) return;
    finish_few<EPI>(p, sl, 0, scale, nb, active, wave, ks, nbi, reinterpret_cast<float*>(rings), acc0, acc1, acc2, acc3, pairs);
  } else {
    RowScales rs{};
    if (active) {
      typedef typename std::conditional<epi_dense(EPI), FullActs, FullActsAhead>::type Acts;
      stream_block_behind<EPI, Acts, Ring>(p, sl, 0, nb, share.c0, share.c1, lane, ring, acc0, acc1, acc2, acc3, wait);
      rs = row_scales<true>(sl, nb, lane & 15);
    }
    if (!wait.there) return;
    finish_block<EPI, true, RING_BYTES / 4>(p, sl, rs, nb, active, ks, nbi, reinterpret_cast<float*>(rings), acc0, acc1, acc2, acc3);
  }
}
template <int EPI, bool A8, bool SPLIT, class Ring = W3Ring>
__device__ __forceinline__ void stream_workgroup(const StreamParams& p, const Slot& sl, int bx, uint8_t* rings) {
  NoWait none;
  stream_workgroup<EPI, A8, SPLIT, Ring>(p, sl, bx, rings, none);
}

template <int EPI, bool A8, bool SPLIT = false, int BITS = 3>  // BITS: the tile layout's (two-bit matrices have their own)
__global__ __launch_bounds__(1024) void w3_stream_kernel(StreamParams p) {
  extern __shared__ __align__(16) uint8_t rings[];
  const Slot sl = slot_of<EPI>(p, blockIdx.y);
  if (sl.rows <= 0) return;  // a slot the plan did not fill: the whole workgroup leaves
  stream_workgroup<EPI, A8, SPLIT, W3RingOf<2, BITS>>(p, sl, blockIdx.x, rings);
}

// A dense call of one slot whose blocks are fewer than half the compute units: PARTS workgroups a 64-row block,
// each its 4 / PARTS 16-row tiles (of the block's loads it asks only for those with its tiles' dwords, and the ones that two
// parts need come from the L2 the second time: a block's workgroups are on one die). The sums and their order are those of
// the one workgroup. What bounds the undivided launch is the expansion on a third of the device.
template <bool A8, bool FEW, int T0, int T1>
__device__ __forceinline__ void part_block(const StreamParams& p, const Slot& sl, int nb, const WaveShare& share, int lane, int wave, uint8_t* rings) {
  f32x4_t acc0 = {0.f, 0.f, 0.f, 0.f}, acc1 = acc0, acc2 = acc0, acc3 = acc0;
  uint8_t* ring = rings + wave * RING_BYTES;
  if constexpr (FEW) {
    const float scale = sl.rs[nb * 64 + lane];
    if constexpr (A8) {
      stream_block<EPI_DENSE, FewActs8Part<T0, T1>, W3RingPart<2, T0, T1>>(p, sl, 0, nb, share.c0, share.c1, lane, ring, acc0, acc1, acc2, acc3);
    } else {
      stream_block<EPI_DENSE, FewActsPart<T0, T1>, W3RingPart<2, T0, T1>>(p, sl, 0, nb, share.c0, share.c1, lane, ring, acc0, acc1, acc2, acc3);
    }
    finish_few<EPI_DENSE>(p, sl, 0, scale, nb, true, wave, share.ks, 0, reinterpret_cast<float*>(rings), acc0, acc1, acc2, acc3, FewPairs{}, FewScales{},
                          T0, T1);
  } else {
    if constexpr (A8) {
      stream_block<EPI_DENSE, FullActs8Part<T0, T1>, W3RingPart<2, T0, T1>>(p, sl, 0, nb, share.c0, share.c1, lane, ring, acc0, acc1, acc2, acc3);
    } else {
      stream_block<EPI_DENSE, FullActsPart<T0, T1>, W3RingPart<2, T0, T1>>(p, sl, 0, nb, share.c0, share.c1, lane, ring, acc0, acc1, acc2, acc3);
    }
    // finish_block for these tiles: the splits' sums through LDS, added in split order, an accumulator register a split and turn
    const RowScales rs = row_scales<true>(sl, nb, lane & 15);
    const f32x4_t all[4] = {acc0, acc1, acc2, acc3};
    float* first = reinterpret_cast<float*>(rings);
    float* mine = first + wave * (RING_BYTES / 4);
#pragma unroll
    for (int t = T0; t < T1; t++)
#pragma unroll
      for (int r = 0; r < 4; r++) mine[(t * 4 + r) * 64 + lane] = all[t][r];
    __syncthreads();
    for (int idx = 4 * T0 + share.ks; idx < 4 * T1; idx += p.ks) {
      const int t = idx >> 2, r = idx & 3;
      if (r >= sl.rows) continue;
      float v = 0.f;
      for (int s = 0; s < p.ks; s++) v += first[s * (RING_BYTES / 4) + idx * 64 + lane];
      emit<EPI_DENSE, true>(p, sl, rs, nb, t, r, lane >> 4, lane & 15, v, 0.f);
    }
  }
}
template <bool A8, bool FEW, int PARTS>
__global__ __launch_bounds__(1024) void w3_part_kernel(StreamParams p) {
  extern __shared__ __align__(16) uint8_t rings[];
  const int die = blockIdx.x & 7, local = blockIdx.x >> 3, part = local % PARTS, nb = local / PARTS * 8 + die;
  if (nb >= p.n_blocks) return;
  const Slot sl = slot_of<EPI_DENSE>(p, 0);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const WaveShare share = wave_share(p, wave);
  if constexpr (PARTS == 2) {
    if (part == 0) part_block<A8, FEW, 0, 2>(p, sl, nb, share, lane, wave, rings); else part_block<A8, FEW, 2, 4>(p, sl, nb, share, lane, wave, rings);
  } else {
    if (part == 0) part_block<A8, FEW, 0, 1>(p, sl, nb, share, lane, wave, rings);
    else if (part == 1) part_block<A8, FEW, 1, 2>(p, sl, nb, share, lane, wave, rings);
    else if (part == 2) part_block<A8, FEW, 2, 3>(p, sl, nb, share, lane, wave, rings);
    else part_block<A8, FEW, 3, 4>(p, sl, nb, share, lane, wave, rings);
  }
}

// A body that hands over the sums of every K split of the dense launch (`Splits`) by itself: at a split's last chunk they go to the
// workgroup's table in LDS and start again from zero, so that a wavefront may take several splits in a row and the table holds what as many
// wavefronts would have left. A lane's part of a split, FEW: the four rows' sums over the four groups, (0 + 1) + (2 + 3) as finish_few adds them, of
// one tile (two tiles: of two rows of one) - else what its accumulators hold. Written as statements of their own: the compiler would have the
// LDS-direct loads of the weights wait ahead of its own LDS stores.
template <bool FEW, int TILES>
constexpr int split_bytes() { return (FEW ? 256 : 1024) * TILES; }
template <class Acts, bool FEW, int T0, int T1>
struct Splits : Acts {
  uint32_t to;          // LDS byte address of the lane's part of the split under way
  int left, base, more; // chunks it has left; chunks of the next ones, one more in the next `more` of them
  __device__ __forceinline__ void hand_over(f32x4_t& acc0, f32x4_t& acc1, f32x4_t& acc2, f32x4_t& acc3) {
    f32x4_t* const all[4] = {&acc0, &acc1, &acc2, &acc3};
    if constexpr (!FEW) {
#pragma unroll
      for (int t = T0; t < T1; t++) asm volatile("ds_write_b128 %0, %1 offset:%2" ::"v"(to), "v"(*all[t]), "n"(1024 * (t - T0)));
    } else {
      float pair[4][2];  // [row][pair of tiles]: lanes' quarters: groups 0 + 1 of the first and of the second tile, groups 2 + 3 of them
#pragma unroll
      for (int r = 0; r < 4; r++)
#pragma unroll
        for (int t = T0; t < T1; t += 2) {
          const auto x = __builtin_amdgcn_permlane16_swap(__float_as_uint((*all[t])[r]), __float_as_uint((*all[t + 1])[r]), false, false);
          pair[r][(t - T0) / 2] = __uint_as_float(x[0]) + __uint_as_float(x[1]);
        }
      auto whole = [](float a, float b) {  // quarters: a's two tiles, b's two tiles
        const auto x = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
        return __uint_as_float(x[0]) + __uint_as_float(x[1]);
      };
      if constexpr (T1 - T0 == 4) {
        const f32x4_t v = {whole(pair[0][0], pair[0][1]), whole(pair[1][0], pair[1][1]), whole(pair[2][0], pair[2][1]), whole(pair[3][0], pair[3][1])};
        asm volatile("ds_write_b128 %0, %1" ::"v"(to), "v"(v));
      } else {
        typedef __attribute__((ext_vector_type(2))) float f32x2_t;
        const f32x2_t v = {whole(pair[0][0], pair[1][0]), whole(pair[2][0], pair[3][0])};
        asm volatile("ds_write_b64 %0, %1" ::"v"(to), "v"(v));
      }
    }
    acc0 = f32x4_t{0.f, 0.f, 0.f, 0.f};
    acc1 = acc2 = acc3 = acc0;
    to += split_bytes<FEW, T1 - T0>();
    more--;
    left = base + (more > 0 ? 1 : 0);
  }
  template <int ODD, bool MORE2, bool MORE1, class C>
  __device__ __forceinline__ void step(const C& ch, int i, f32x4_t& acc0, f32x4_t& acc1, f32x4_t& acc2, f32x4_t& acc3, const Slot& sl) {
    Acts::template step<ODD, MORE2, MORE1>(ch, i, acc0, acc1, acc2, acc3, sl);
    if (--left == 0) hand_over(acc0, acc1, acc2, acc3);  // uniform
  }
};

// The gate | up projection of a dense SwiGLU block of at most sixteen rows together with what its 3-bit down projection takes: silu(gate) * up
// as the BF16 tensor expression rounds it, then E4M3 codes and a scale a 32-group (p.oq, p.oq_scale [rows, p.out_stride]).
// A workgroup holds the 64-row block of gate rows and the block of up rows of the same 64 columns of h (PARTS 2: half of either's
// tiles, 32 columns), so that a pair of values meets in LDS and neither leaves the compute unit. K has the p.ks splits of the dense launch, `run` of
// them one after the other a wavefront (Splits), and the sums are the dense launch's bit for bit.
struct GateUp {
  int half_blocks, pair_blocks;  // h's 64-column blocks; > 0: gate and up alternate in runs of that many blocks
  int ways, run;                 // wavefronts a block; splits a wavefront: ways * run == p.ks
};
template <bool FEW, int T0, int T1>
__device__ __forceinline__ void gate_up_block(const StreamParams& p, const GateUp& g, const Slot& sl, int gate, int up, int column0, int lane, int wave,
                                              uint8_t* rings) {
  constexpr int TILES = T1 - T0, GROUPS = TILES / 2, SPLIT = split_bytes<FEW, TILES>() / 4;  // 32-column groups of h; floats a split
  const int q = lane >> 4, r16 = lane & 15;
  const int second = wave >= g.ways ? 1 : 0, s0 = (wave - second * g.ways) * g.run, s1 = s0 + g.run;  // the wavefront's splits
  const int nb = second ? up : gate, c0 = s0 * p.chunks_base + min(s0, p.chunks_rem), c1 = s1 * p.chunks_base + min(s1, p.chunks_rem);
  // the row scales of what this lane will add up, asked for ahead of the chunks: FEW: lanes 0 .. 31 a group's gate rows, 32 .. 63 its
  // up rows; else both tiles of both
  f32x4_t scale0 = {0.f, 0.f, 0.f, 0.f}, scale1 = scale0;  // of the first and the second group (an array of both would be indexed, and so held in memory)
  auto scales_of = [&](f32x4_t& to, int t) {
    if constexpr (FEW) {
      to.x = sl.rs[(lane < 32 ? gate : up) * 64 + 16 * t + (lane & 31)];
    } else {
#pragma unroll
      for (int j = 0; j < 4; j++) to[j] = sl.rs[(j < 2 ? gate : up) * 64 + 16 * (t + (j & 1)) + r16];
    }
  };
  scales_of(scale0, T0);
  if constexpr (GROUPS == 2) scales_of(scale1, T0 + 2);
  uint8_t* ring = rings + wave * RING_BYTES;
  const float* const sums = reinterpret_cast<const float*>(rings + 2 * g.ways * RING_BYTES);  // [gate, up][split]
  f32x4_t acc0 = {0.f, 0.f, 0.f, 0.f}, acc1 = acc0, acc2 = acc0, acc3 = acc0;
  auto stream = [&](auto acts, auto ring_of) {
    acts.to = (uint32_t)(uintptr_t)(lds_ptr_t)(rings + 2 * g.ways * RING_BYTES) + (second * p.ks + s0) * (4 * SPLIT) + lane * (FEW ? 4 * TILES : 16);
    acts.base = p.chunks_base;
    acts.more = p.chunks_rem - s0;
    acts.left = acts.base + (acts.more > 0 ? 1 : 0);
    stream_block<EPI_DENSE, decltype(acts), decltype(ring_of)>(p, sl, 0, nb, c0, c1, lane, ring, acc0, acc1, acc2, acc3, acts);
  };
  if constexpr (TILES == 4) {
    stream(Splits<typename std::conditional<FEW, FewActs, FullActs>::type, FEW, T0, T1>{}, W3Ring{});
  } else {
    stream(Splits<typename std::conditional<FEW, FewActsPart<T0, T1>, FullActsPart<T0, T1>>::type, FEW, T0, T1>{}, W3RingPart<2, T0, T1>{});
  }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // (hand_over's writes: the compiler does not count them)
  __syncthreads();
  // a unit of work: accumulator register r of a group's tiles (FEW: row r of the slot)
  for (int unit = wave; unit < (FEW ? sl.rows : min(4, sl.rows)) * GROUPS; unit += 2 * g.ways) {  // uniform
    const int r = GROUPS == 2 ? unit >> 1 : unit, gr = GROUPS == 2 ? unit & 1 : 0, t = 2 * gr;
    const f32x4_t scale = gr ? scale1 : scale0;
    if constexpr (FEW) {
      const int tile = t + (q & 1);
      const float* at = sums + (lane < 32 ? 0 : p.ks * SPLIT) + (TILES == 4 ? (tile * 16 + r16) * 4 + r : (((r & 1) * 2 + tile) * 16 + r16) * 2 + (r >> 1));
      float v = 0.f;
      for (int s = 0; s < p.ks; s++, at += SPLIT) v += *at;
      const float y = through_bf16(v * scale.x), other = __shfl_xor(y, 32);
      const float h = silu_chain(lane < 32 ? y : other, lane < 32 ? other : y);
      float amax = row16_max(fabsf(h));
      amax = fmaxf(amax, __shfl_xor(amax, 16));
      if (lane < 32) store_quantized(p, r, column0 + 32 * gr + lane, h, amax, lane == 0);
    } else {
      const int i = 4 * q + r;
      float v[4] = {0.f, 0.f, 0.f, 0.f};
      const float *first = sums + (t * 64 + lane) * 4 + r, *other = first + p.ks * SPLIT;
      for (int s = 0; s < p.ks; s++, first += SPLIT, other += SPLIT) v[0] += first[0], v[1] += first[256], v[2] += other[0], v[3] += other[256];
      if (i >= sl.rows) continue;  // whole rows of lanes
#pragma unroll
      for (int j = 0; j < 4; j++) v[j] = through_bf16(v[j] * scale[j]);
      const float h0 = silu_chain(v[0], v[2]), h1 = silu_chain(v[1], v[3]);
      const float amax = row16_max(fmaxf(fabsf(h0), fabsf(h1)));
      store_quantized(p, i, column0 + 32 * gr + r16, h0, amax, r16 == 0);
      store_quantized(p, i, column0 + 32 * gr + 16 + r16, h1, amax, false);
    }
  }
}
constexpr int GATE_UP_WAYS = 4;  // at most
template <bool FEW, int PARTS>
__global__ __launch_bounds__(64 * 2 * GATE_UP_WAYS) void w3_fc_gate_up_kernel(StreamParams p, GateUp g) {
  extern __shared__ __align__(16) uint8_t rings[];
  const int die = blockIdx.x & 7, local = blockIdx.x >> 3, part = local % PARTS, b = PARTS == 1 ? (int)blockIdx.x : local / PARTS * 8 + die;
  if (b >= g.half_blocks) return;
  const int gate = g.pair_blocks ? b / g.pair_blocks * 2 * g.pair_blocks + b % g.pair_blocks : b, up = gate + (g.pair_blocks ? g.pair_blocks : g.half_blocks);
  const Slot sl = slot_of<EPI_DENSE>(p, 0);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if constexpr (PARTS == 1) {
    gate_up_block<FEW, 0, 4>(p, g, sl, gate, up, 64 * b, lane, wave, rings);
  } else if (part == 0) {
    gate_up_block<FEW, 0, 2>(p, g, sl, gate, up, 64 * b, lane, wave, rings);
  } else {
    gate_up_block<FEW, 2, 4>(p, g, sl, gate, up, 64 * b + 32, lane, wave, rings);
  }
}

// One token from its router logits: fc1 with the routing inside it, so that the call has no launch for routing and plan.
// Every wavefront of the launch routes the row for itself (about three microseconds in which it could not have known
// its expert anyway; the logits are 2 KB): lane s then holds selection s, slot s is that expert with the token's one
// row, and the slot after the last selection is the shared expert's. The first wavefront of the first workgroup also
// writes what the caller and the next launch read: ids, weights, and the slot table and pair list in the plan's format
// (in selection order: every slot has one row, so no order is better). The activation row is row 0 whatever a slot's
// pair index says: the launch passes a row stride of 0.
template <int EPI>
__global__ __launch_bounds__(1024) void w3_fc1_route_one_kernel(StreamParams p, RouteParams route, int e_lo, int e_n, int shared_slot, int32_t* plan,
                                                                int32_t* order) {
  extern __shared__ __align__(16) uint8_t rings[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const bool writer = blockIdx.x == 0 && blockIdx.y == 0 && wave == 0;
  const int id = route.per <= 8 ? route_row<false, 8>(route, 0, lane, writer) : route_row<false, 16>(route, 0, lane, writer);
  const int local = id - e_lo;
  const bool here = lane < route.k && local >= 0 && local < e_n;  // an expert of another rank's range has no slot
  if (writer) {
    const int kept = __popcll(__ballot(here));
    if (lane < route.k || lane == shared_slot) {
      int32_t* entry = plan + PLAN_HEADER + 4 * lane;
      entry[0] = lane == shared_slot ? -1 : here ? local : 0;
      entry[1] = lane;
      entry[2] = lane == shared_slot || here ? 1 : 0;
      entry[3] = 0;
      order[lane] = lane;  // a selection's pair index is its own; the shared expert's row follows the pairs
    }
    if (lane == 0) {
      plan[0] = route.k + (shared_slot >= 0 ? 1 : 0);
      plan[1] = plan[2] = kept;
    }
  }
  const int slot = blockIdx.y;
  int expert = -1;
  if (slot != shared_slot) {
    if (!__builtin_amdgcn_readlane((int)here, slot)) return;  // uniform over the workgroup
    expert = __builtin_amdgcn_readlane(local, slot);
  }
  stream_workgroup<EPI, false, false, W3RingCached>(p, make_slot(p, slot, expert, slot, 1), blockIdx.x, rings);
}

// fc1 and fc2 of a routed call in ONE launch, so that fc2's workgroups fill the compute units that fc1's last, partly
// empty round of workgroups leaves idle (and no launch boundary lies between the two). The grid is one-dimensional:
// first every fc1 workgroup (slot-major, the slot table's order), then every fc2 workgroup. A slot's fc2 needs all of
// the slot's h, that is all `groups1` fc1 workgroups of the slot: each of those, once its h is in memory (write-through
// stores, waited for), adds one to the slot's arrival counter (plan_done: zero from the plan), and the slot's fc2
// workgroups wait for the counter behind the requests of their first weights (one wavefront polls with loads that bypass the L2, the
// others stand at a barrier: SlotWait). What fc2 then reads of h it reads with ordinary loads: the lines were written through to
// memory before the count, and this compute die's L2 cannot hold an older copy of them, because every launch starts
// with its L2 invalidated and no workgroup of this launch reads a slot's h before the slot's count is complete (h rows
// are whole 256-byte multiples on 256-byte boundaries, so no line of h is shared with anything read earlier).
// fc2 workgroups cannot starve fc1: the hardware starts a grid's workgroups in index order, so when an fc2 workgroup
// waits, every fc1 workgroup has started, and an fc1 workgroup waits for nothing. HIP does not promise that order;
// should it ever fail to hold, await_count's bound ends the wait, the workgroup records HB_FAULT_WAIT in the
// workspace's fault word (hb_workspace_status reads it) and leaves without storing anything. hb_tune("moe_fused", 2)
// runs the two layers as two launches, which wait for nothing. Same sums in the same order either way: the same bits.
//
// Order of the grid: slot-major, fc2 of a slot `lag` slots behind its fc1 - fc1(0) .. fc1(lag - 1), then fc1(s), fc2(s -
// lag) for s = lag .., then the last `lag` slots' fc2. With `lag` about the slots whose workgroups fill the device once,
// a slot's fc2 workgroups are started when its fc1 workgroups have had a workgroup's lifetime to finish: they rarely
// wait, and fc1 and fc2 workgroups of different lengths run side by side instead of in rounds that start and end
// together. The slots a call does not fill (the table's upper bound is far above them: every pair could name another
// expert) come last in this order, fc1 and fc2 alike, so their workgroups, short as they are, hold nobody back.
template <int EPI1, bool SPLIT>
__global__ __launch_bounds__(1024) void w3_fc12_kernel(StreamParams p1, StreamParams p2, int groups1, int groups2, int slots, int lag) {
  extern __shared__ __align__(16) uint8_t rings[];
  __shared__ int outcome;
  const Fc12Place at = fc12_place(blockIdx.x, groups1, groups2, slots, lag);
  const int slot = at.slot;
  const int64_t t0 = p1.trace ? (int64_t)wall_clock64() : 0;
  int64_t t1 = 0;
  int rows = 0;
  if (at.is_fc1) {
    const Slot sl = slot_of<EPI1>(p1, slot);
    if (sl.rows <= 0) return;
    rows = sl.rows;
    stream_workgroup<EPI1, false, SPLIT>(p1, sl, at.index, rings);
    fc12_arrive(p1, slot);
  } else {
    const Slot sl = slot_of<EPI_FC2>(p2, slot);
    if (sl.rows <= 0) return;
    rows = sl.rows;
    SlotWait wait(p2, slot, &outcome, p1.trace != nullptr);
    stream_workgroup<EPI_FC2, false, false>(p2, sl, at.index, rings, wait);
    if (!wait.there) return;  // h is not known to be complete: this workgroup's outputs stay as they were
    t1 = wait.ended;
  }
  if (p1.trace && threadIdx.x == 0 && (int64_t)blockIdx.x < p1.trace_records) {  // measurement hook: start, end of the wait, end (100 MHz ticks), rows
    int64_t* rec = p1.trace + 4 * (int64_t)blockIdx.x;
    rec[0] = t0;
    rec[1] = t1;
    rec[2] = (int64_t)wall_clock64();
    rec[3] = rows | (at.is_fc1 ? 1 << 16 : 0);
  }
}

// One token (a decode step): fc2 and the combine in one launch. A workgroup owns a 64-row block of the output; each of
// its first `slots` wavefronts takes one slot of the plan (an expert the token chose, or the shared expert) through all
// of K on the four-row body, adds its groups as finish_few does without a K split, and leaves the slot's 64 outputs in
// LDS under the pair's selection index; with a gate, four more wavefronts meanwhile make its dot product. The first
// wavefront then runs the combine's chain, a column a lane. Every sum is the one the two separate launches make (fc2
// with one K split, then moe_combine_kernel), so the bits are theirs; what goes away is the round trip of the pair
// outputs through memory and a launch.
constexpr int ONE_GATE_WAVES = 4;  // the gate's dot product is laid out over 256 threads
constexpr int ONE_MAX_WAVES = 16;

// One wavefront's product over all of K for the tiles T0 .. T1 - 1 of block row nb (the others' accumulators: zero).
template <int T0, int T1>
__device__ __forceinline__ void one_token_tiles(const StreamParams& p, const Slot& sl, int row0, int nb, int lane, uint8_t* ring, f32x4_t (&acc)[4]) {
  if constexpr (T0 == 0 && T1 == 4) {
    stream_block<EPI_FC2, FewActs, W3RingCached>(p, sl, row0, nb, 0, p.chunks, lane, ring, acc[0], acc[1], acc[2], acc[3]);
  } else {
    stream_block<EPI_FC2, FewActsPart<T0, T1>, W3RingPart<0, T0, T1>>(p, sl, row0, nb, 0, p.chunks, lane, ring, acc[0], acc[1], acc[2], acc[3]);
  }
}

// PARTS: the workgroups a 64-row block (1, 2 or 4), each taking 4 / PARTS of its four 16-row tiles - the same sums a
// column, over more compute units: a workgroup's wavefronts expand only their tiles' codes (a slot's whole K is four
// chunks of 204 VALU instructions a wavefront otherwise, and a workgroup's ten or eleven wavefronts share four SIMDs)
// and ask only for the 16-byte loads those tiles' dwords lie in (one or two of a chunk's three).
template <int PARTS>
__global__ __launch_bounds__(1024) void w3_fc2_combine_one_kernel(StreamParams p, CombineParams c, int slots) {
  extern __shared__ __align__(16) uint8_t rings[];  // a ring a streaming wavefront, then ys [topk + 1][64], then the gate's four partial sums
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nb = blockIdx.x / PARTS, part = blockIdx.x % PARTS, q = lane >> 4, r16 = lane & 15;
  float* ys = reinterpret_cast<float*>(rings + slots * RING_BYTES);
  float* red = ys + (p.topk + 1) * 64;
  // the chain's operands, a selection a lane, asked for now; a pair whose expert is not local has no slot: its place
  // in ys is never written and never read
  float w_mine = 0.f;
  bool keep_mine = false;
  if (wave == 0 && lane < p.topk) {
    const int e = c.ids[lane] - c.e_lo;
    keep_mine = e >= 0 && e < c.e_n;
    w_mine = c.weights[lane];
  }
  if (wave >= slots) {  // only with a gate
    combine_gate_partial(c.x, c.gate_vec, c.hx, 0, (int)threadIdx.x - 64 * slots, red);
  } else {
    const Slot sl = slot_of<EPI_FC2>(p, wave);
    if (sl.rows > 0) {  // uniform over the wavefront
      const float scale = sl.rs[nb * 64 + lane];
      float* mine = reinterpret_cast<float*>(rings + wave * RING_BYTES);
      for (int row0 = 0; row0 < sl.rows; row0 += FEW_ROWS) {  // more than one row: the caller named an expert twice
        f32x4_t acc[4];
#pragma unroll
        for (int t = 0; t < 4; t++) acc[t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        FewPairs pairs;
        pairs.ask(p, sl, row0);
        uint8_t* ring = reinterpret_cast<uint8_t*>(mine);
        if (PARTS == 1) {
          one_token_tiles<0, 4>(p, sl, row0, nb, lane, ring, acc);
        } else if (PARTS == 2) {
          if (part == 0) one_token_tiles<0, 2>(p, sl, row0, nb, lane, ring, acc); else one_token_tiles<2, 4>(p, sl, row0, nb, lane, ring, acc);
        } else {
          if (part == 0) one_token_tiles<0, 1>(p, sl, row0, nb, lane, ring, acc);
          else if (part == 1) one_token_tiles<1, 2>(p, sl, row0, nb, lane, ring, acc);
          else if (part == 2) one_token_tiles<2, 3>(p, sl, row0, nb, lane, ring, acc);
          else one_token_tiles<3, 4>(p, sl, row0, nb, lane, ring, acc);
        }
#pragma unroll
        for (int t = 0; t < 4; t++) {
          mine[(t * 4 + 0) * 64 + lane] = acc[t].x;
          mine[(t * 4 + 1) * 64 + lane] = acc[t].y;
          mine[(t * 4 + 2) * 64 + lane] = acc[t].z;
          mine[(t * 4 + 3) * 64 + lane] = acc[t].w;
        }
        __builtin_amdgcn_wave_barrier();  // the lanes of one wavefront: its LDS operations execute in program order
        const int rows = min(FEW_ROWS, sl.rows - row0);
        for (int r = 0; r < rows; r++) {
          const float* at = mine + (q * 4 + r) * 64 + r16;
          float v = 0.f;
          v += (at[0] + at[16]) + (at[32] + at[48]);
          ys[min(pairs.of(r), p.topk) * 64 + lane] = v * scale;  // lane (q, r16) is column 16 q + r16 of the block; the shared expert's row follows the pairs
        }
        __builtin_amdgcn_wave_barrier();  // read before the next pass's blocks land in the ring
      }
    }
  }
  __syncthreads();
  if (wave != 0) return;
  // Every lane runs the chain and only the store is narrowed to this workgroup's tiles: the chain reads its operands
  // from lanes 0 .. topk - 1, and what a lane outside the execution mask holds of a value computed earlier is not
  // defined (the compiler may compute it after the branch that narrowed the mask).
  float v = 0.f;
  for (int s = 0; s < p.topk; s++) {
    const bool keep = __builtin_amdgcn_readlane((int)keep_mine, s) != 0;
    const float w = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, w_mine), s));
    v = fmaf(keep ? w : 0.f, keep ? ys[s * 64 + lane] : 0.f, v);
  }
  if (c.shared) v = combine_shared(v, c.gate_vec ? combine_gate_value(red) : 1.0f, ys[p.topk * 64 + lane]);
  if (PARTS == 1 || q / (4 / PARTS) == part) c.out[nb * 64 + lane] = f32_to_bf16_bits(v);  // lane (q, r16) is column 16 q + r16
}

// ---------------------------------------------------------------------------------- the panel kernel's W3 formats
// A fragment's eight weights: two selectors and two permutes give their E4M3 codebook bytes, which are expanded times the
// group's E4M3 scale (a 4-bit significand times a 4-bit one: exact in BF16); the FP32 row scale stays in the epilogue.
template <int BITS>
struct TileW3 {
  typedef W3RingOf<2, BITS> Ring;
  typedef typename Ring::Chunk Chunk;
  static constexpr int BLOCK_BYTES = Ring::BLOCK_BYTES;
  static constexpr bool PER_ROW = true;
  // For search_panel: a chunk of a pair of wavefronts takes this much longer than NVFP4's; and up to this many row tiles the
  // registers of two eight-wavefront workgroups fit a compute unit (the pair of them is 10 % faster than whole rounds say).
  static constexpr float EXPAND_US = 0.45f;
  static constexpr int BESIDE_TILES = 3;
  // A routed call's slots of at most this many rows run on the weight stream's bodies, a wavefront a block over all of K. With
  // one product a fragment the panel's expansion to scaled BF16 (four conversions, eight multiplications and four roundings a
  // fragment) bounds the slot: 100 to 107 cycles a fragment and SIMD, two wavefronts. The stream's bodies convert
  // without the scale and fold it into the FP32 sums (four conversions, four multiply-adds; up to four rows one): 84. Skewed
  // routing of 10 of 512 experts (2048, 512), where 218 of 377 slots are such: the layer of 1024 rows 205 -> 187 us, 1543
  // 251 -> 234, 2048 296 -> 271; even routing at the same sizes unchanged. A ring of four slots with the activations as far
  // ahead gave nothing: what the wavefronts wait for is each other's issue slots.
  static constexpr int LOW_ROWS = 22, MIDDLE_ROWS = 60, MIDDLE_ROWS_LARGE = 72, HIGH_ROWS = 88;  // panel_height's lines
  static constexpr int LIGHT_ROWS = ROWS_PER_SLOT;
  template <int EPI, class Wait>
  static __device__ __forceinline__ void light(const StreamParams& p, const Slot& sl, int group, uint8_t* lds, Wait& wait) {
    static_assert(BITS == 3 || epi_dense(EPI), "routed experts are three-bit");
    if constexpr (BITS == 3) stream_workgroup<EPI, false, false, Ring>(p, sl, group, lds, wait);
  }
  struct Part {
    uint32_t lo, hi;  // codebook bytes of weights 0 .. 3 and 4 .. 7
    float scale;
  };
  template <int NT, int S>
  static __device__ __forceinline__ Part open(const Chunk& ch, const Slot& sl) {
    uint32_t sel[8];
    chunk_selectors<NT>(ch, sel);  // the six the step does not use fold away
    return Part{__builtin_amdgcn_perm(sl.lut_hi, sl.lut_lo, sel[2 * S]), __builtin_amdgcn_perm(sl.lut_hi, sl.lut_lo, sel[2 * S + 1]),
                __builtin_amdgcn_cvt_f32_fp8(chunk_scales<NT>(ch), S)};
  }
#define HB_W3_CVT "v_cvt_scalef32_pk_f32_fp8"
  template <int K, bool AFTER_VALU>  // a product, then values 2 K, 2 K + 1 of the part
  static __device__ __forceinline__ void product_pair(f32x4_t& acc, const u32x4_t& w, const u32x4_t& a, const Part& part, uint32_t& out) {
    if constexpr (K == 0 && AFTER_VALU) HB_PANEL_PRODUCT_PAIR("s_nop 1\n\t", HB_W3_CVT, "", acc, out, w, part.lo, part.scale, a);
    if constexpr (K == 0 && !AFTER_VALU) HB_PANEL_PRODUCT_PAIR("", HB_W3_CVT, "", acc, out, w, part.lo, part.scale, a);
    if constexpr (K == 1) HB_PANEL_PRODUCT_PAIR("", HB_W3_CVT, " op_sel:[1,0,0]", acc, out, w, part.lo, part.scale, a);
    if constexpr (K == 2) HB_PANEL_PRODUCT_PAIR("", HB_W3_CVT, "", acc, out, w, part.hi, part.scale, a);
    if constexpr (K == 3) HB_PANEL_PRODUCT_PAIR("", HB_W3_CVT, " op_sel:[1,0,0]", acc, out, w, part.hi, part.scale, a);
  }
  template <int K, bool AFTER_VALU>  // a product, then the first half of that
  static __device__ __forceinline__ void product_first(f32x4_t& acc, const u32x4_t& w, const u32x4_t& a, const Part& part, panel_two_t& two) {
    if constexpr (K == 0 && AFTER_VALU) HB_PANEL_PRODUCT_FIRST("s_nop 1\n\t", HB_W3_CVT, "", acc, two, w, part.lo, part.scale, a);
    if constexpr (K == 0 && !AFTER_VALU) HB_PANEL_PRODUCT_FIRST("", HB_W3_CVT, "", acc, two, w, part.lo, part.scale, a);
    if constexpr (K == 1) HB_PANEL_PRODUCT_FIRST("", HB_W3_CVT, " op_sel:[1,0,0]", acc, two, w, part.lo, part.scale, a);
    if constexpr (K == 2) HB_PANEL_PRODUCT_FIRST("", HB_W3_CVT, "", acc, two, w, part.hi, part.scale, a);
    if constexpr (K == 3) HB_PANEL_PRODUCT_FIRST("", HB_W3_CVT, " op_sel:[1,0,0]", acc, two, w, part.hi, part.scale, a);
  }
  template <int K>
  static __device__ __forceinline__ void pair_alone(const Part& part, uint32_t& out) {
    if constexpr (K == 0) HB_PANEL_PAIR_ALONE(HB_W3_CVT, "", out, part.lo, part.scale);
    if constexpr (K == 1) HB_PANEL_PAIR_ALONE(HB_W3_CVT, " op_sel:[1,0,0]", out, part.lo, part.scale);
    if constexpr (K == 2) HB_PANEL_PAIR_ALONE(HB_W3_CVT, "", out, part.hi, part.scale);
    if constexpr (K == 3) HB_PANEL_PAIR_ALONE(HB_W3_CVT, " op_sel:[1,0,0]", out, part.hi, part.scale);
  }
};

// A dense call: the stream's passes (one a sixteen rows) run side by side while their blocks do not fill the device, and the
// few rows of a second pass are nearly free. Measured, stream and panel: 5120 x 5120 (80 blocks) 48 rows 10.9 and 15.0 us,
// 64 rows 16.3 and 14.2, 128 rows 22.6 and 16.8; 8192 x 2048 32 rows 7.6 and 8.8, 48 rows 9.8 and 9.0; 51200 x 2048 17 rows
// 20.6 and 20.3, 48 rows 30.7 and 22.8; 51200 x 5120 128 rows 195 and 70.
constexpr int PANEL_W3_ROWS = 20, PANEL_W3_BLOCKS = 300;

// ---------------------------------------------------------------------------------------------------- host side
struct Tuning {  // hb_tune's knobs: relaxed atomics, so a knob set from one thread while another launches is a plain race-free read
  std::atomic<int> w3_tile{0}, w3_few{0}, w3_ksplit{0}, w3_nbw{0}, moe_fc1_ksplit{0}, moe_fc1_nbw{0}, moe_fc2_ksplit{0}, moe_fc2_nbw{0}, moe_one{0}, moe_split{0}, moe_fused{0}, moe_lag{0}, moe_one_parts{0};
};
static Tuning g_tune;

// Launch one W3 stream. `busy_slots` is the caller's estimate of the slots that will have rows (the grid covers
// `slots`, the upper bound); K is split until the launch has a few thousand wavefronts.
struct Launch {
  int ks, nbw;  // 0: chosen here
};

// Chooses the workgroup shape of a launch (p.ks, p.nbw and what follows from them).
static int shape_stream(StreamParams& p, int64_t busy_slots, Launch want) {
  pick_shape(p.n_blocks, p.chunks, busy_slots, 8192, &p.ks, &p.nbw);
  if (want.ks) {
    p.ks = want.ks;
    if (!want.nbw) p.nbw = 1;
  }
  if (want.nbw) p.nbw = want.nbw;
  if (p.ks * p.nbw > 16 || p.ks > p.chunks) return HB_EINVAL;
  set_split(p);
  p.no_few = g_tune.w3_few == 2;  // every slot takes the sixteen-row body
  return HB_OK;
}

// The shape of a dense call of one slot. A wavefront's start and the exchange cost about as much as two chunks of its K, the
// expansion of a chunk more with each row. Measured, replayed graphs of calls on cycled weights, the general rule and this one
// (us, blocks x chunks): twelve rows, K split eight ways: 40 x 12 8.9 and 5.0, 160 x 12 8.9 and 5.2, 640 x 24 17.8 and 16.9,
// 400 x 7 9.4 and 7.0; up to four rows, at least four: 160 x 4 5.2 and 3.5, 400 x 7 6.9 and 5.4, 640 x 12 9.5 and 8.3. The general rule
// stays where its workgroups fit the device better:
// - up to four rows of 257 to 512 blocks, from eight chunks: two blocks a workgroup all start at once, and four ways
//   took 1.00 to 1.12 times as long (one row of 300 x 10: 1.08, 512 x 10 1.07, 400 x 12 0.99);
// - past three blocks a compute unit: four ways or eight of 2374 x 4 and 2374 x 8 chunks at twelve rows took 1.21 and 1.16 times as
//   long (1200 x 8 0.93). From twelve rows one form gains there: up to four blocks a compute unit, some have four of them
//   whichever way they are dealt out, and runs of four start a quarter of the workgroups: sixteen rows of 800 x 16 0.94,
//   1024 x 16 0.95, two-bit 1000 x 20 0.95; twelve and thirteen rows 0.96 to 1.01, two-bit 0.95 to 1.01 (770 to 1024 blocks,
//   12 to 31 chunks). With fewer rows it is even (eight rows 0.98 to 1.05), and with fewer blocks or more the runs leave units
//   idle: 768 x 24 1.14, 1200 x 24 1.42.
constexpr int COMPUTE_UNITS = 256, RUN_ROWS = 12;
static void shape_dense(StreamParams& p) {
  const bool few = p.m <= FEW_ROWS && !p.no_few;
  auto split = [&](int most) {  // at least as many ways as the general rule
    while (p.ks < most && 2 * p.ks <= p.chunks) p.ks *= 2;
    p.nbw = p.ks >= 4 ? 1 : p.nbw;
  };
  if (few) {
    if (p.n_blocks < 3 * COMPUTE_UNITS && (p.n_blocks <= COMPUTE_UNITS || p.n_blocks > 2 * COMPUTE_UNITS || p.chunks < 8)) split(4);
  } else if (p.n_blocks <= 3 * COMPUTE_UNITS) {
    split(8);
  } else if (p.n_blocks <= 4 * COMPUTE_UNITS && p.m >= RUN_ROWS && p.chunks >= 12 && p.chunks < 32) {
    p.ks = 2;
    p.nbw = 4;
  }
  set_split(p);
}

// Blocks up to which a dense call of one slot gives a block's tiles to two workgroups (up to half of them: to four).
// 5120 x 5120 at one row 7.7 -> 6.4 us; the dense block at four rows (its down projection is 5120 x 25600) 50.5 -> 46.7. Five to
// sixteen rows, replayed graphs, eight rows: 1024 x 4096 7.8 -> 5.5 us, 4096 x 5120 9.5 -> 6.6, 8192 x 5120 9.9 -> 7.5; the dense
// block of ten rows (4096, 8192), whose down projection takes E4M3 activations, 31.2 -> 24.8.
constexpr int PARTS_BLOCKS = 128;
// The shape of a dense call of one slot whose shape nobody forces; whether it runs in parts.
static bool shape_one_slot(StreamParams& p, int bits) {
  const bool few = p.m <= FEW_ROWS, parted = bits == 3 && p.n_blocks <= PARTS_BLOCKS && !(few && p.no_few);
  if (!p.aq && !(parted && few)) shape_dense(p);
  return parted;
}
template <int EPI>
static int launch_stream(StreamParams& p, int64_t slots, int64_t busy_slots, Launch want, hipStream_t stream, int bits = 3) {
  if (int e = shape_stream(p, busy_slots, want)) return e;
  if constexpr (EPI == EPI_DENSE) {
    const bool few = p.m <= FEW_ROWS;
    if (slots == 1 && !want.ks && !want.nbw && !p.a2 && shape_one_slot(p, bits)) {
      p.nbw = 1;
      const int parts = p.n_blocks <= PARTS_BLOCKS / 2 ? 4 : 2;
      const dim3 blocks((unsigned)((p.n_blocks + 7) / 8 * 8 * parts));
      auto launch = [&](auto kernel) { HB_LAUNCH(kernel, blocks, dim3(64 * p.ks), (size_t)p.ks * RING_BYTES, stream, p); };
      if (few) {
        if (p.aq) {
          parts == 4 ? launch(w3_part_kernel<true, true, 4>) : launch(w3_part_kernel<true, true, 2>);
        } else {
          parts == 4 ? launch(w3_part_kernel<false, true, 4>) : launch(w3_part_kernel<false, true, 2>);
        }
      } else if (p.aq) {
        parts == 4 ? launch(w3_part_kernel<true, false, 4>) : launch(w3_part_kernel<true, false, 2>);
      } else {
        parts == 4 ? launch(w3_part_kernel<false, false, 4>) : launch(w3_part_kernel<false, false, 2>);
      }
      return HB_OK;
    }
  }
  const dim3 grid((unsigned)((p.n_blocks + p.nbw - 1) / p.nbw), (unsigned)slots);
  const int waves = p.ks * p.nbw;
  const size_t lds = (size_t)waves * RING_BYTES;
  if (bits == 2) {  // dense calls only: the reference's two-plane matrices are dense linears (its draft head)
    if constexpr (epi_dense(EPI)) {
      if (p.aq) {
        HB_LAUNCH((w3_stream_kernel<EPI, true, false, 2>), grid, dim3(64 * waves), lds, stream, p);
      } else {
        HB_LAUNCH((w3_stream_kernel<EPI, false, false, 2>), grid, dim3(64 * waves), lds, stream, p);
      }
      return HB_OK;
    }
    return HB_EINVAL;
  }
  if (p.aq) {
    HB_LAUNCH((w3_stream_kernel<EPI, true>), grid, dim3(64 * waves), lds, stream, p);
  } else if (p.a2 && !p.no_few) {
    HB_LAUNCH((w3_stream_kernel<EPI, false, true>), grid, dim3(64 * waves), lds, stream, p);
  } else {
    HB_LAUNCH((w3_stream_kernel<EPI, false>), grid, dim3(64 * waves), lds, stream, p);
  }
  return HB_OK;
}

}  // namespace hb

using namespace hb;

#ifndef HB_NO_DEBUG_HOOKS
extern "C" int hb_tune(const char* key, int value) {
  if (!key) return HB_ENULL;
  struct {
    const char* name;
    std::atomic<int>* slot;
  } table[] = {{"w3_tile", &g_tune.w3_tile}, {"w3_few", &g_tune.w3_few}, {"w3_ksplit", &g_tune.w3_ksplit},           {"w3_nbw", &g_tune.w3_nbw},
               {"moe_fc1_ksplit", &g_tune.moe_fc1_ksplit}, {"moe_fc1_nbw", &g_tune.moe_fc1_nbw},
               {"moe_fc2_ksplit", &g_tune.moe_fc2_ksplit}, {"moe_fc2_nbw", &g_tune.moe_fc2_nbw}, {"moe_one", &g_tune.moe_one}, {"moe_split", &g_tune.moe_split}, {"moe_fused", &g_tune.moe_fused}, {"moe_lag", &g_tune.moe_lag}, {"moe_one_parts", &g_tune.moe_one_parts}};
  for (auto& t : table)
    if (!strcmp(t.name, key)) {
      if (value < 0 || value > 16) return HB_EINVAL;
      *t.slot = value;
      return HB_OK;
    }
  if (moe_tune(key, value) == HB_OK) return HB_OK;
  return nvfp4_tune(key, value);
}
#endif

extern "C" int hb_w3_gemm(const void* x, int m, const void* tiled, const float* row_scale, int64_t lut, int n, int k, int bits, void* y, void* stream) {
  if (!x || !tiled || !row_scale || !y) return HB_ENULL;
  if (m <= 0 || n <= 0 || k <= 0 || n % W3_BLOCK_ROWS || k % W3_CHUNK || (bits != 2 && bits != 3)) return HB_EINVAL;
  if (!aligned(x, 16) || !aligned(tiled, 16) || !aligned(row_scale, 4) || !aligned(y, 2)) return HB_EINVAL;
  StreamParams p{};
  p.w = static_cast<const uint8_t*>(tiled);
  p.rows = row_scale;
  p.lut_lo = (uint32_t)((uint64_t)lut & 0xffffffffu);
  p.lut_hi = (uint32_t)((uint64_t)lut >> 32);
  p.n_blocks = n / W3_BLOCK_ROWS;
  p.chunks = k / W3_CHUNK;
  p.a = static_cast<const uint16_t*>(x);
  p.a_stride = k;
  p.m = m;
  p.out = y;
  p.out_stride = n;
  if (panel_takes(m, k) && panel_writes(y, false) && (g_tune.w3_tile == 1 || (g_tune.w3_tile == 0 && m > PANEL_W3_ROWS && (int64_t)p.n_blocks * ((m + ROWS_PER_SLOT - 1) / ROWS_PER_SLOT) >= PANEL_W3_BLOCKS))) {
    const PanelForce force{g_tune.w3_ksplit, g_tune.w3_nbw, 0};
    if (int e = bits == 2 ? launch_panel<TileW3<2>, EPI_DENSE>(p, cut_panel<TileW3<2>>(m, p.n_blocks, p.chunks, 0, force), nullptr, as_stream(stream))
                          : launch_panel<TileW3<3>, EPI_DENSE>(p, cut_panel<TileW3<3>>(m, p.n_blocks, p.chunks, 0, force), nullptr, as_stream(stream)))
      return e;
    return launch_status();
  }
  const int64_t slots = (m + ROWS_PER_SLOT - 1) / ROWS_PER_SLOT;
  if (slots > 65535) return HB_EINVAL;
  if (int e = launch_stream<EPI_DENSE>(p, slots, slots, Launch{g_tune.w3_ksplit, g_tune.w3_nbw}, as_stream(stream), bits)) return e;
  return launch_status();
}

extern "C" int hb_w3_quant_groups(const void* x, int64_t m, int k, void* q, float* scales, void* stream) {
  if (!x || !q || !scales) return HB_ENULL;
  if (m <= 0 || k <= 0 || k % 32) return HB_EINVAL;
  if (!aligned(x, 16) || !aligned(q, 8) || !aligned(scales, 4)) return HB_EINVAL;
  moe_launch_quant_groups(QuantJob{static_cast<const uint16_t*>(x), m * k / 8, static_cast<uint8_t*>(q), scales, 0, 0}, as_stream(stream));
  return launch_status();
}

extern "C" int hb_w3_quant_rows(const void* x, int64_t m, int k, void* q, float* scales, void* stream) {
  if (!x || !q || !scales) return HB_ENULL;
  if (m <= 0 || m > 0x7fffffff || k <= 0 || k % 8) return HB_EINVAL;
  if (!aligned(x, 16) || !aligned(q, 8) || !aligned(scales, 4)) return HB_EINVAL;
  moe_launch_quant_rows(static_cast<const uint16_t*>(x), m, k, static_cast<uint8_t*>(q), scales, as_stream(stream));
  return launch_status();
}

static int check_e4m3(const void* xq, const float* x_scale, int m, const void* tiled, const float* row_scale, int n, int k, int bits, const void* y) {
  if (!xq || !x_scale || !tiled || !row_scale || !y) return HB_ENULL;
  if (m <= 0 || n <= 0 || k <= 0 || n % W3_BLOCK_ROWS || k % W3_CHUNK || (int64_t)m * (k / 32) > 0xffffffffll || (bits != 2 && bits != 3)) return HB_EINVAL;
  if (!aligned(xq, 8) || !aligned(x_scale, 8) || !aligned(tiled, 16) || !aligned(row_scale, 4) || !aligned(y, 2)) return HB_EINVAL;
  return ((int64_t)m + ROWS_PER_SLOT - 1) / ROWS_PER_SLOT > 65535 ? HB_EINVAL : HB_OK;
}

extern "C" int hb_w3_gemm_e4m3(const void* xq, const float* x_scale, int m, const void* tiled, const float* row_scale, int64_t lut, int n, int k,
                               int bits, void* y, void* stream) {
  if (int e = check_e4m3(xq, x_scale, m, tiled, row_scale, n, k, bits, y)) return e;
  StreamParams p{};
  p.w = static_cast<const uint8_t*>(tiled);
  p.rows = row_scale;
  p.lut_lo = (uint32_t)((uint64_t)lut & 0xffffffffu);
  p.lut_hi = (uint32_t)((uint64_t)lut >> 32);
  p.n_blocks = n / W3_BLOCK_ROWS;
  p.chunks = k / W3_CHUNK;
  p.aq = static_cast<const uint8_t*>(xq);
  p.aq_scale = x_scale;
  p.a_stride = k;
  p.m = m;
  p.out = y;
  p.out_stride = n;
  const int64_t slots = ((int64_t)m + ROWS_PER_SLOT - 1) / ROWS_PER_SLOT;
  if (int e = launch_stream<EPI_DENSE>(p, slots, slots, Launch{g_tune.w3_ksplit, g_tune.w3_nbw}, as_stream(stream), bits)) return e;
  return launch_status();
}

// The dense SwiGLU block on its 3-bit copies. Gate | up, the SiLU product and its E4M3 rounding are one launch up to sixteen rows
// (w3_fc_gate_up_kernel), which keeps gate | up out of memory and costs two launches' starts and ends less: the block (5120, 25600) of four rows
// 52.7 -> 50.1 us, (4096, 8192) of one and sixteen 19.1 -> 15.5 and 28.6 -> 26.9, (1024, 1024) of four 10.5 -> 8.1 (replayed graphs on cycled weights).
// Its splits of K are the dense launch's, so that its bits are; a wavefront takes `run` of them, and what it hands over between them costs 2 to
// 4 % of the launch (a K split of its own, which a block of 400 x 40 had in two ways for eight, gave 41.8 us where this gives 42.8).
// Its shape, by h's 64-column blocks B and the chunks of K; swept over 16 to 1024 blocks, 8 to 64 chunks, one to sixteen rows, times of the three
// launches (1.0):
// - up to 128 blocks half of them a workgroup, four wavefronts a block: 0.77 to 0.98. The gate | up of up to 64 blocks alone is dealt out
//   by quarters of a block, and where K is long that weighs more: up to four rows 1.01 to 1.05 of 16 and 32 x 40 and 64 x 64 (48 x 40 0.96, 128 x 64
//   0.90), above 1.0 to 1.17 of up to 64 x 40, from twelve rows 1.0 to 1.05 of up to 64 x 24 and 1.05 of 128 x 64;
// - up to 256 whole blocks, four wavefronts: 0.81 to 0.93 (more than four rows past 40 chunks: the sums leave no room for the rings);
// - up to 384 halves, two wavefronts: 0.86 to 0.98 up to four rows; above 0.96 to 0.99 of 8 chunks and 0.98 to 1.05 from 16;
// - up to 512 whole blocks, two wavefronts: 0.88 to 0.97; more than four rows below 32 chunks, where a workgroup's sums leave room
//   for a second one: 0.89 to 0.94, else 1.04 to 1.1;
// - past them, up to four rows, by what their last round leaves idle: whole blocks 0.93 to 0.98 where it is nearly full (700, 1024), else halves 0.88
//   to 0.98 (540, 600, 800; whole 0.9 to 1.05) below 32 chunks and 0.96 to 1.02 above; more rows whole blocks below 24 chunks 0.92 to
//   1.0, else 0.97 to 1.2.
struct GateUpShape {
  int parts, ways;  // parts 0: three launches
};
static GateUpShape gate_up_shape(int m, int blocks, int chunks) {
  const bool few = m <= FEW_ROWS;
  GateUpShape s{1, 2};
  if (blocks <= 128) {
    s = GateUpShape{2, 4};
    if (few ? chunks >= 32 && blocks <= chunks : blocks <= 64 ? chunks >= (m >= 12 ? 24 : 32) : m >= 12 && chunks >= 48) s.parts = 0;
  } else if (blocks <= 256) {
    s = GateUpShape{1, 4};
  } else if (blocks <= 384) {
    s = GateUpShape{few || chunks < 16 ? 2 : 0, 2};
  } else if (!few) {
    if (chunks >= (blocks <= 512 ? 32 : 24)) s.parts = 0;
  } else if (blocks > 512) {
    const int last = blocks % COMPUTE_UNITS;  // workgroups of whole blocks in the last round
    if (last && last < COMPUTE_UNITS * 5 / 8) s.parts = chunks < 32 ? 2 : 0;
  }
  while (s.ways > 1 && (few ? 2 : 1) * s.ways > chunks) s.ways /= 2;  // a wavefront's start costs about two chunks of the four-row body
  return s;
}

extern "C" int hb_w3_mlp(const void* x, int m, const void* gate_up, const float* gate_up_rows, int64_t gate_up_lut, int inter, int hidden, int gate_up_bits,
                         int pairs, const void* down, const float* down_rows, int64_t down_lut, int n, int down_bits, void* scratch, size_t scratch_bytes, void* y,
                         void* stream) {
  if (!x || !gate_up || !gate_up_rows || !down || !down_rows || !scratch || !y) return HB_ENULL;
  if (m <= 0 || inter <= 0 || inter > 0x3fffffff || hidden <= 0 || inter % W3_CHUNK || hidden % W3_CHUNK || pairs < 0 || (pairs && (pairs % 32 || inter % pairs)) || (gate_up_bits != 2 && gate_up_bits != 3)) return HB_EINVAL;
  if (!aligned(x, 16) || !aligned(gate_up, 16) || !aligned(gate_up_rows, 4) || !aligned(scratch, 16)) return HB_EINVAL;
  if (scratch_bytes < HB_W3_MLP_SCRATCH_BYTES((size_t)m, (size_t)inter)) return HB_EWORKSPACE;
  uint8_t* hq = static_cast<uint8_t*>(scratch);
  float* h_scale = reinterpret_cast<float*>(hq + (size_t)m * inter);
  if (int e = check_e4m3(hq, h_scale, m, down, down_rows, n, inter, down_bits, y)) return e;  // ahead of the first launch
  const int blocks = inter / W3_BLOCK_ROWS;
  StreamParams p{};
  p.w = static_cast<const uint8_t*>(gate_up);
  p.rows = gate_up_rows;
  p.lut_lo = (uint32_t)((uint64_t)gate_up_lut & 0xffffffffu);
  p.lut_hi = (uint32_t)((uint64_t)gate_up_lut >> 32);
  p.n_blocks = 2 * blocks;
  p.chunks = hidden / W3_CHUNK;
  p.a = static_cast<const uint16_t*>(x);
  p.a_stride = hidden;
  p.m = m;
  p.oq = hq;
  p.oq_scale = h_scale;
  p.out_stride = inter;
  const bool forced = g_tune.w3_tile || g_tune.w3_few || g_tune.w3_ksplit || g_tune.w3_nbw;  // (a shape of the dense launch's own)
  const bool few = m <= FEW_ROWS, fits = m <= ROWS_PER_SLOT && gate_up_bits == 3 && pairs % W3_BLOCK_ROWS == 0 && blocks <= 0xffffff && !forced;
  const GateUpShape shape = fits ? gate_up_shape(m, blocks, p.chunks) : GateUpShape{0, 1};
  GateUp g{blocks, pairs / W3_BLOCK_ROWS, 1, 1};
  size_t lds = 0;
  if (shape.parts) {
    if (int e = shape_stream(p, 1, Launch{0, 0})) return e;
    shape_one_slot(p, 3);  // the dense launch's splits of K
    g.ways = std::min(shape.ways, p.ks);
    g.run = p.ks / g.ways;
    const int split = few ? split_bytes<true, 4>() : split_bytes<false, 4>();
    lds = (size_t)2 * g.ways * RING_BYTES + (size_t)2 * p.ks * split / shape.parts;
  }
  if (shape.parts && lds <= PANEL_LDS) {
    const dim3 grid((unsigned)(shape.parts == 1 ? blocks : (blocks + 7) / 8 * 8 * 2)), block(64 * 2 * g.ways);
    auto launch = [&](auto kernel) { HB_LAUNCH(kernel, grid, block, lds, as_stream(stream), p, g); };
    if (few) {
      shape.parts == 1 ? launch(w3_fc_gate_up_kernel<true, 1>) : launch(w3_fc_gate_up_kernel<true, 2>);
    } else {
      shape.parts == 1 ? launch(w3_fc_gate_up_kernel<false, 1>) : launch(w3_fc_gate_up_kernel<false, 2>);
    }
  } else {
    uint16_t* both = reinterpret_cast<uint16_t*>(hq + (size_t)m * inter / 8 * 9);
    if (int e = hb_w3_gemm(x, m, gate_up, gate_up_rows, gate_up_lut, 2 * inter, hidden, gate_up_bits, both, stream)) return e;
    if (int e = hb_silu_mul_quant_groups(both, m, inter, pairs, 1, hq, h_scale, stream)) return e;
  }
  return hb_w3_gemm_e4m3(hq, h_scale, m, down, down_rows, down_lut, n, inter, down_bits, y, stream);
}

// ------------------------------------------------------------------------------------------------ routed experts
namespace {

int check_experts(const hb_w3_experts* ex) {
  if (!ex) return HB_ENULL;
  if (!ex->fc1 || !ex->fc1_rows || !ex->fc2 || !ex->fc2_rows) return HB_ENULL;
  if (ex->experts <= 0 || ex->hidden <= 0 || ex->inter <= 0 || ex->hidden_out <= 0) return HB_EINVAL;
  const int n1 = ex->gated ? 2 * ex->inter : ex->inter;
  if (ex->hidden % W3_CHUNK || ex->inter % W3_CHUNK || n1 % W3_BLOCK_ROWS || ex->hidden_out % W3_BLOCK_ROWS) return HB_EINVAL;
  if (!aligned(ex->fc1, 16) || !aligned(ex->fc2, 16) || !aligned(ex->fc1_rows, 4) || !aligned(ex->fc2_rows, 4)) return HB_EINVAL;
  return HB_OK;
}

// plan -> fc1 -> fc2 (-> combine, when `combine` is given): `out_pairs` receives fc2's per-pair outputs (the
// workspace's y unless the caller wants the pairs themselves). One token's fc2 and combine are one launch.
struct Routing {  // set: the chain routes the logits itself into the caller's ids / weights
  TopkRoute top;
  int32_t* ids;
  float* weights;
  const BudgetRoute* budget = nullptr;  // ... under a budget (`top` is then unused)
};

int run_experts(const hb_w3_experts* ex, const hb_w3_experts* shared, const void* x, const int32_t* ids, int m, int topk,
                const MoeWorkspace& ws, void* out_pairs, int pairs_bf16, hipStream_t stream, int experts_total, const Routing* route = nullptr,
                bool e4m3 = false, const CombineParams* combine = nullptr) {
  const int64_t pairs = (int64_t)m * topk, named = experts_named(experts_total, ex->base, ex->experts);
  const int shared_rows = shared ? m : 0;
  // A dense contraction once an expert sees some rows: the panel kernel's higher slots (E4M3 activations: the stream only).
  // The stream pays for a pass a sixteen rows, the panel for longer workgroups, which a call of few experts does not fill: `fill` is fc1's, a
  // slot an expert. The lines lie where neither even nor skewed routing loses. Measured, even and (skewed) routing, stream and panel, the
  // whole layer in us, experts (hidden, inter), fill: 512 (2048, 512), 2048, 5 rows an expert 175 and 166 (117 and 99), 9 rows 198 and 192 (167 and 125);
  // 256 (2560, 768), 1536, 5 rows 164 and 155 (122 and 101); 300 (1280, 384), 900, 5 rows 72 and 72 (59 and 61), 7 rows 77 and 76 (69 and 64); 180 (1664, 384), 540,
  // 5 rows 70 and 70 (61 and 62), 7 rows 72 and 71 (67 and 63); 96 (2560, 768), 576, 11 rows 93 and 96 (97 and 92), 18 rows 128 and 111 (125 and 106); 64
  // (2048, 512), 256, 22 rows 74 and 78 (73 and 75), 27 rows 81 and 78 (81 and 78); 128 (1024, 256), 256, 18 rows 55 and 55 (54 and 54), 22 rows 61 and 59 (57 and 59),
  // 27 rows 65 and 60 (64 and 61). A range of the experts sees its share of the pairs only.
  // Few wide experts fill it with fc1 and not with fc2, whose workgroups (`fill2`) are then few and as long as their K: 96 (1024, 3072), fill2 a chunk of K 16, 9 rows
  // 96 and 103 (103 and 111), 16 rows 130 and 129 (136 and 128); 64 (1536, 4096), 12, 7 rows 123 and 121 (126 and 130); 48 (2048, 8192), 6, 5 rows 204 and 212 (201 and 229),
  // 9 rows 240 and 230 (270 and 253); 128 (2048, 4096), 32, 5 rows 263 and 267 (244 and 243); 32 (2048, 4096), 8, 15 rows 115 and 112 (115 and 121); 16 (2048, 8192),
  // 2, 20 rows 150 and 155 (147 and 174), 40 rows 222 and 192 (223 and 215); 24 (2048, 6144), 4, 20 rows 162 and 156 (149 and 166), 30 rows 218 and 167 (219 and 196).
  const int64_t fill = (int64_t)ex->experts * (((ex->gated ? 2 : 1) * ex->inter / W3_BLOCK_ROWS + 3) / 4), fill2 = (int64_t)ex->experts * ((ex->hidden_out / W3_BLOCK_ROWS + 3) / 4);
  const int chunks2 = ex->inter / W3_CHUNK;
  const int rows_min = fill >= 500 && ex->experts < 150 && fill2 < 5 * chunks2                   ? 24
                       : fill >= 1500                                                            ? fill2 >= 30 * chunks2 ? 5 : ex->hidden >= 1536 ? 9 : 14
                       : fill >= 500                                                             ? ex->experts >= 150 ? 7 : 16
                       : ex->experts < named                                                     ? 48
                                                                                                 : 26;
  const bool dense = !e4m3 && panel_takes(m, ex->hidden) && panel_takes(pairs + shared_rows, ex->inter) && panel_writes(out_pairs, !pairs_bf16) &&
                     (g_tune.w3_tile == 1 || (g_tune.w3_tile == 0 && pairs >= rows_min * named));
  const int tiles = panel_height<TileW3<3>>(pairs, named, ex->experts, shared_rows, (ex->gated ? 2 : 1) * ex->inter / W3_BLOCK_ROWS), slot_rows = dense ? 16 * tiles : ROWS_PER_SLOT;
  // Under a budget the table ends behind the experts the selection can name: the launches' grids reach over all of it, and a
  // workgroup without rows is not free (40 rows of 10, a cap of 60 of 512 experts: 53.5 us before, 53.2 so). What a call of
  // these pairs is refused for, and how its launches split K, go by the whole table: the bits of the same ids without a budget.
  const int64_t whole = moe_max_slots(pairs, ex->experts, shared_rows, std::min(slot_rows, PANEL_REFUSED_ROWS));
  if (whole > PANEL_MAX_SLOTS) return HB_EINVAL;
  if (route && route->budget) {
    if (int e = moe_check_budget(*route->budget, m, topk)) return e;
  }
  const int64_t distinct = route && route->budget ? budget_distinct(*route->budget, m, ex->experts) : ex->experts;
  const int64_t slots = moe_max_slots(pairs, (int)distinct, shared_rows, slot_rows);
  // E4M3 activations: x is rounded by further workgroups of the plan's launch, h in fc1's epilogue
  // weight-only on the stream: x also in its two-plane form, for the slots of at most two rows (fc1 on the FP8 matrix cores)
  const bool split = !e4m3 && !dense && g_tune.moe_split == 1 && g_tune.w3_few != 2;
  const QuantJob xjob = split ? QuantJob{static_cast<const uint16_t*>(x), 0, ws.x2, ws.x2s, m, ex->hidden}
                              : QuantJob{static_cast<const uint16_t*>(x), (int64_t)m * ex->hidden / 8, ws.xq, ws.xs, 0, 0};
  const QuantJob* job = e4m3 || split ? &xjob : nullptr;
  // one token from its logits, a slot a selection, and fc2 + combine as one launch after it: fc1 routes for itself
  const bool route_in_fc1 = route && !route->budget && !route->top.slots && m == 1 && combine && !e4m3 && !split && !dense && topk <= 63 && slots == topk + shared_rows &&
                            slots + (combine->gate_vec && combine->shared ? ONE_GATE_WAVES : 0) <= ONE_MAX_WAVES && g_tune.moe_one == 0 &&
                            moe_check_route(m, route->top.e, topk) == HB_OK;
  if (route_in_fc1) {
    // (nothing to launch here)
  } else if (route && route->budget) {
    if (e4m3) return HB_EINVAL;  // weight-only
    if (job) moe_launch_quant_groups(*job, stream);  // the selection's launch carries no rounding job: the two-plane form of x in a launch of its own
    // the rows' candidates rest where the pair outputs will go: the selection has read them before fc2 writes
    if (int e = moe_launch_budget_plan(*route->budget, m, topk, route->ids, route->weights, ex->base, ex->experts, shared_rows, ws, ws.y, stream, slot_rows))
      return e;
  } else if (route) {
    if (int e = moe_launch_route_plan(route->top, m, topk, route->ids, route->weights, ex->base, ex->experts, shared_rows, ws, stream, slot_rows, job))
      return e;
  } else if (int e = moe_launch_plan(ids, pairs, ex->base, ex->experts, shared_rows, ws, stream, slot_rows, job)) {
    return e;
  }
  const int n1 = ex->gated ? 2 * ex->inter : ex->inter;
  const int64_t est = pairs < 2 * ex->experts ? (pairs + 1) / 2 + (shared_rows + 15) / 16 : whole;  // rough number of busy slots
  StreamParams p{};
  p.w = static_cast<const uint8_t*>(ex->fc1);
  p.expert_bytes = (int64_t)hb_w3_tiled_bytes(n1, ex->hidden, 3);
  p.rows = ex->fc1_rows;
  p.expert_rows = n1;
  p.lut_lo = (uint32_t)((uint64_t)ex->fc1_lut & 0xffffffffu);
  p.lut_hi = (uint32_t)((uint64_t)ex->fc1_lut >> 32);
  if (shared) {
    p.w_shared = static_cast<const uint8_t*>(shared->fc1);
    p.rows_shared = shared->fc1_rows;
    p.lut_lo_shared = (uint32_t)((uint64_t)shared->fc1_lut & 0xffffffffu);
    p.lut_hi_shared = (uint32_t)((uint64_t)shared->fc1_lut >> 32);
  }
  p.n_blocks = n1 / W3_BLOCK_ROWS;
  p.chunks = ex->hidden / W3_CHUNK;
  p.a = static_cast<const uint16_t*>(x);
  p.a_stride = ex->hidden;
  p.plan = ws.plan;
  p.order = ws.order;
  p.topk = topk;
  p.pairs = (int)pairs;
  p.out = ws.h;
  p.out_stride = ex->inter;
  StreamParams f2 = p;
  f2.w = static_cast<const uint8_t*>(ex->fc2);
  f2.expert_bytes = (int64_t)hb_w3_tiled_bytes(ex->hidden_out, ex->inter, 3);
  f2.rows = ex->fc2_rows;
  f2.expert_rows = ex->hidden_out;
  f2.lut_lo = (uint32_t)((uint64_t)ex->fc2_lut & 0xffffffffu);
  f2.lut_hi = (uint32_t)((uint64_t)ex->fc2_lut >> 32);
  if (shared) {
    f2.w_shared = static_cast<const uint8_t*>(shared->fc2);
    f2.rows_shared = shared->fc2_rows;
    f2.lut_lo_shared = (uint32_t)((uint64_t)shared->fc2_lut & 0xffffffffu);
    f2.lut_hi_shared = (uint32_t)((uint64_t)shared->fc2_lut >> 32);
  }
  f2.n_blocks = ex->hidden_out / W3_BLOCK_ROWS;
  f2.chunks = ex->inter / W3_CHUNK;
  f2.a = ws.h;
  f2.a_stride = ex->inter;
  f2.out = out_pairs;
  f2.out_stride = ex->hidden_out;
  f2.out_bf16 = pairs_bf16;
  if (dense && g_tune.moe_fused != 2 && fc12_apart(p) && (g_tune.moe_fused == 1 || panel_together(p, f2, ex->experts, tiles))) {
    if (int e = ex->gated ? launch_panel_fc12<TileW3<3>, EPI_FC1_GATED>(p, f2, ws.plan, tiles, slots, m, pairs + shared_rows, g_tune.moe_lag, stream)
                          : launch_panel_fc12<TileW3<3>, EPI_FC1_RELU2>(p, f2, ws.plan, tiles, slots, m, pairs + shared_rows, g_tune.moe_lag, stream))
      return e;
    if (combine) moe_launch_combine(*combine, stream);
    return launch_status();
  }
  if (dense) {
    if (int e = ex->gated ? launch_panel_routed<TileW3<3>, EPI_FC1_GATED>(p, tiles, slots, m, stream) : launch_panel_routed<TileW3<3>, EPI_FC1_RELU2>(p, tiles, slots, m, stream)) return e;
    if (int e = launch_panel_routed<TileW3<3>, EPI_FC2>(f2, tiles, slots, pairs + shared_rows, stream)) return e;
    if (combine) moe_launch_combine(*combine, stream);
    return launch_status();
  }
  Launch l1{g_tune.moe_fc1_ksplit, g_tune.moe_fc1_nbw}, l2{g_tune.moe_fc2_ksplit, g_tune.moe_fc2_nbw};
  // Decode batches of a few rows to a couple of dozen leave the device partly empty under the general rule (K split 4,
  // one block a workgroup; fc2: four blocks). Measured on the fused launch at hidden 2048 / intermediate 512: up to
  // about 48 busy slots fc1 with K split 2 on two blocks and fc2 with K split 4 is 3 - 5 % faster a step, from 64 to
  // 128 busy slots both with K split 2 on two blocks 3 %; beyond that the general rule wins.
  const bool unset = !l1.ks && !l1.nbw && !l2.ks && !l2.nbw;
  if (unset && !e4m3 && m > 1 && g_tune.moe_fused != 2 && p.chunks >= 8 && f2.chunks >= 4) {
    if (est <= 48) {
      l1 = Launch{2, 2};
      l2 = Launch{4, 1};
    } else if (est >= 64 && est <= 128) {
      l1 = Launch{2, 2};
      l2 = Launch{2, 2};
    }
  }
  if (e4m3) {  // x and h go through the activation rounding: x_q -> fc1 -> h_q -> fc2
    p.aq = ws.xq;
    p.aq_scale = ws.xs;
    p.oq = ws.hq;
    p.oq_scale = ws.hs;
    f2.aq = ws.hq;
    f2.aq_scale = ws.hs;
  }
  if (split) {
    p.a2 = ws.x2;
    p.a2_scale = ws.x2s;
  }
  // more than one token, weight-only: fc1 and fc2 as one launch when their workgroups have the same shape
  if (!e4m3 && m > 1 && g_tune.moe_fused != 2 && fc12_apart(p)) {
    StreamParams q1 = p, q2 = f2;
    if (shape_stream(q1, est, l1) == HB_OK && shape_stream(q2, est, l2) == HB_OK && q1.ks * q1.nbw == q2.ks * q2.nbw) {
      const int groups1 = (q1.n_blocks + q1.nbw - 1) / q1.nbw, groups2 = (q2.n_blocks + q2.nbw - 1) / q2.nbw;
      const int64_t total = slots * (groups1 + groups2);
      if (total <= 0x7fffffff) {
        moe_await_slots(q1, q2, ws.plan, slots, groups1);
        q1.trace = moe_trace_buffer(&q1.trace_records);
        const int waves = q1.ks * q1.nbw;
        // about the slots whose workgroups fill the device once (four workgroups of four wavefronts a compute unit)
        const int lag_tuned = g_tune.moe_lag.load();
        const int lag = (int)std::min<int64_t>(slots, lag_tuned ? 8 * lag_tuned : std::max(8, 2304 / (groups1 + groups2)));
        const bool use_split = q1.a2 && !q1.no_few;
        auto launch = [&](auto kernel) { HB_LAUNCH(kernel, dim3((unsigned)total), dim3(64 * waves), (size_t)waves * RING_BYTES, stream, q1, q2, groups1, groups2, (int)slots, lag); };
        if (ex->gated) {
          use_split ? launch(w3_fc12_kernel<EPI_FC1_GATED, true>) : launch(w3_fc12_kernel<EPI_FC1_GATED, false>);
        } else {
          use_split ? launch(w3_fc12_kernel<EPI_FC1_RELU2, true>) : launch(w3_fc12_kernel<EPI_FC1_RELU2, false>);
        }
        if (combine) moe_launch_combine(*combine, stream);
        return launch_status();
      }
    }
  }
  if (route_in_fc1) {
    StreamParams q = p;
    if (int e = shape_stream(q, est, l1)) return e;
    q.a_stride = 0;  // every slot's row is the token's
    RouteParams rp{};
    rp.logits = static_cast<const float*>(route->top.logits);
    rp.half = route->top.half;
    rp.stride = route->top.e;
    rp.e = route->top.e;
    rp.k = topk;
    rp.per = (route->top.e + 63) / 64;
    rp.steps = 1;
    rp.pad_id = route->top.e;
    rp.ids = route->ids;
    rp.weights = route->weights;
    const dim3 grid((unsigned)((q.n_blocks + q.nbw - 1) / q.nbw), (unsigned)slots);
    const int waves = q.ks * q.nbw;
    auto launch = [&](auto kernel) {
      HB_LAUNCH(kernel, grid, dim3(64 * waves), (size_t)waves * RING_BYTES, stream, q, rp, ex->base, ex->experts, shared ? topk : -1, ws.plan, ws.order);
    };
    ex->gated ? launch(w3_fc1_route_one_kernel<EPI_FC1_GATED>) : launch(w3_fc1_route_one_kernel<EPI_FC1_RELU2>);
  } else if (int e = ex->gated ? launch_stream<EPI_FC1_GATED>(p, slots, est, l1, stream) : launch_stream<EPI_FC1_RELU2>(p, slots, est, l1, stream)) {
    return e;
  }
  int fc2_ks = l2.ks, fc2_nbw;
  if (!fc2_ks) pick_shape(f2.n_blocks, f2.chunks, est, 8192, &fc2_ks, &fc2_nbw);
  // one token, and a separate fc2 would not split K either: the fused launch makes the same sums
  const int one_waves = (int)slots + (combine && combine->gate_vec && combine->shared ? ONE_GATE_WAVES : 0);
  // (its chain hands the selections' weights from lane to lane: at most 64 of them)
  if (combine && m == 1 && topk <= 64 && !e4m3 && one_waves <= ONE_MAX_WAVES && fc2_ks == 1 && g_tune.moe_one != 2) {
    f2.ks = 1;
    f2.nbw = 1;
    set_split(f2);
    // the workgroups a 64-row block: as many as leave the launch within about the device's compute units
    const int parts = g_tune.moe_one_parts ? g_tune.moe_one_parts.load() : f2.n_blocks <= 64 ? 4 : f2.n_blocks <= 128 ? 2 : 1;
    const size_t lds = (size_t)slots * RING_BYTES + (topk + 1) * 256 + 16;
    if (parts == 4) {
      HB_LAUNCH(w3_fc2_combine_one_kernel<4>, dim3(4u * (unsigned)f2.n_blocks), dim3(64 * one_waves), lds, stream, f2, *combine, (int)slots);
    } else if (parts == 2) {
      HB_LAUNCH(w3_fc2_combine_one_kernel<2>, dim3(2u * (unsigned)f2.n_blocks), dim3(64 * one_waves), lds, stream, f2, *combine, (int)slots);
    } else {
      HB_LAUNCH(w3_fc2_combine_one_kernel<1>, dim3((unsigned)f2.n_blocks), dim3(64 * one_waves), lds, stream, f2, *combine, (int)slots);
    }
    return launch_status();
  }
  if (int e = launch_stream<EPI_FC2>(f2, slots, est, l2, stream)) return e;
  if (combine) moe_launch_combine(*combine, stream);
  return launch_status();
}

}  // namespace

extern "C" size_t hb_w3_moe_workspace_bytes(int m, int topk, const hb_w3_experts* routed, int shared) {
  if (!routed || m <= 0 || topk <= 0 || check_experts(routed) != HB_OK) return 0;
  return moe_carve(nullptr, m, topk, routed->experts, routed->inter, routed->hidden_out, shared, routed->hidden).bytes;
}

#ifndef HB_NO_DEBUG_HOOKS
extern "C" int hb_debug_workspace_layout(int m, int topk, const hb_w3_experts* routed, int shared, int64_t* offsets) {
  if (!routed || !offsets) return HB_ENULL;
  if (m <= 0 || topk <= 0 || check_experts(routed) != HB_OK) return HB_EINVAL;
  char* base = reinterpret_cast<char*>(uintptr_t(1) << 20);  // any address: only differences are returned
  const MoeWorkspace ws = moe_carve(base, m, topk, routed->experts, routed->inter, routed->hidden_out, shared, routed->hidden);
  offsets[0] = reinterpret_cast<char*>(ws.plan) - base;
  offsets[1] = reinterpret_cast<char*>(ws.order) - base;
  offsets[2] = reinterpret_cast<char*>(ws.h) - base;
  offsets[3] = reinterpret_cast<char*>(ws.y) - base;
  offsets[4] = reinterpret_cast<char*>(plan_done(ws.plan, moe_max_slots((int64_t)m * topk, routed->experts, shared ? m : 0))) - base;
  offsets[5] = moe_max_slots((int64_t)m * topk, routed->experts, shared ? m : 0);
  return HB_OK;
}
#endif

extern "C" int hb_w3_moe(const hb_w3_experts* routed, const void* x, const int32_t* ids, const float* weights, int m, int topk, int mode,
                         void* out, void* workspace, size_t workspace_bytes, void* stream) {
  return hb_w3_moe_among(routed, 0, x, ids, weights, m, topk, mode, out, workspace, workspace_bytes, stream);
}

extern "C" int hb_w3_moe_among(const hb_w3_experts* routed, int experts_total, const void* x, const int32_t* ids, const float* weights, int m, int topk,
                               int mode, void* out, void* workspace, size_t workspace_bytes, void* stream) {
  if (int e = check_experts(routed)) return e;
  if (!x || !ids || !weights || !out || !workspace) return HB_ENULL;
  const bool e4m3 = (mode & HB_MOE_E4M3) != 0;
  mode &= ~HB_MOE_E4M3;
  if (m <= 0 || topk <= 0 || mode < HB_MOE_SUM || mode > HB_MOE_PAIRS_BF16) return HB_EINVAL;
  if (!aligned(x, 16) || !aligned(ids, 4) || !aligned(weights, 4) || !aligned(out, 8) || !aligned(workspace, 16)) return HB_EINVAL;
  const MoeWorkspace ws = moe_carve(workspace, m, topk, routed->experts, routed->inter, routed->hidden_out, 0, routed->hidden);
  if (workspace_bytes < ws.bytes) return HB_EWORKSPACE;
  void* pairs_out = mode == HB_MOE_SUM ? static_cast<void*>(ws.y) : out;
  const bool narrow = mode == HB_MOE_SUM && m >= MOE_WIDE_ROWS;  // a summed prefill-sized call: BF16 pair outputs (hibana/model/flashnext/moe.py:186)
  CombineParams c{};
  c.pairs = ws.y;
  c.pairs_bf16 = narrow;
  c.ids = ids;
  c.weights = weights;
  c.e_lo = routed->base;
  c.e_n = routed->experts;
  c.m = m;
  c.topk = topk;
  c.h = routed->hidden_out;
  c.out = static_cast<uint16_t*>(out);
  return run_experts(routed, nullptr, x, ids, m, topk, ws, pairs_out, mode == HB_MOE_PAIRS_BF16 || narrow, as_stream(stream), experts_total, nullptr, e4m3,
                     mode == HB_MOE_SUM ? &c : nullptr);
}

static int moe_layer(const hb_w3_experts* routed, const hb_w3_experts* shared, const float* gate_vec, const void* x, const int32_t* ids,
                     const float* weights, int m, int topk, void* out, void* workspace, size_t workspace_bytes, void* stream,
                     int experts_total, const Routing* route, bool e4m3 = false) {
  if (int e = check_experts(routed)) return e;
  if (shared) {
    if (int e = check_experts(shared)) return e;
    if (shared->hidden != routed->hidden || shared->inter != routed->inter || shared->hidden_out != routed->hidden_out ||
        shared->gated != routed->gated)
      return HB_EINVAL;
  }
  if (!x || !ids || !weights || !out || !workspace) return HB_ENULL;
  if (m <= 0 || topk <= 0) return HB_EINVAL;
  if (!aligned(x, 16) || !aligned(ids, 4) || !aligned(weights, 4) || !aligned(out, 4) || !aligned(workspace, 16) || !aligned(gate_vec, 4)) return HB_EINVAL;
  const MoeWorkspace ws = moe_carve(workspace, m, topk, routed->experts, routed->inter, routed->hidden_out, shared ? 1 : 0, routed->hidden);
  if (workspace_bytes < ws.bytes) return HB_EWORKSPACE;
  // a prefill-sized call keeps its pair outputs (and the shared expert's rows behind them) in BF16, as the reference's
  // layer does from the same size (hibana/model/flashnext/moe.py:186); the shared rows are rounded to BF16 by the combine anyway
  const bool narrow = m >= MOE_WIDE_ROWS;
  CombineParams c{};
  c.pairs = ws.y;
  c.pairs_bf16 = narrow;
  c.ids = ids;
  c.weights = weights;
  if (shared) {
    c.shared = narrow ? static_cast<const void*>(reinterpret_cast<const uint16_t*>(ws.y) + (int64_t)m * topk * routed->hidden_out)
                      : static_cast<const void*>(ws.y + (int64_t)m * topk * routed->hidden_out);
    c.shared_f32 = narrow ? 0 : 1;
    c.shared_stride = routed->hidden_out;
    c.x = static_cast<const uint16_t*>(x);
    c.gate_vec = gate_vec;
    c.hx = routed->hidden;
  }
  c.e_lo = routed->base;
  c.e_n = routed->experts;
  c.m = m;
  c.topk = topk;
  c.h = routed->hidden_out;
  c.out = static_cast<uint16_t*>(out);
  return run_experts(routed, shared, x, ids, m, topk, ws, ws.y, narrow, as_stream(stream), experts_total, route, e4m3, &c);
}

extern "C" int hb_w3_moe_layer(const hb_w3_experts* routed, const hb_w3_experts* shared, const float* gate_vec, const void* x,
                               const int32_t* ids, const float* weights, int m, int topk, void* out, void* workspace,
                               size_t workspace_bytes, void* stream) {
  return moe_layer(routed, shared, gate_vec, x, ids, weights, m, topk, out, workspace, workspace_bytes, stream, 0, nullptr);
}

extern "C" int hb_w3_moe_layer_among(const hb_w3_experts* routed, int experts_total, const hb_w3_experts* shared, const float* gate_vec, const void* x,
                                     const int32_t* ids, const float* weights, int m, int topk, void* out, void* workspace,
                                     size_t workspace_bytes, void* stream) {
  return moe_layer(routed, shared, gate_vec, x, ids, weights, m, topk, out, workspace, workspace_bytes, stream, experts_total, nullptr);
}

extern "C" int hb_w3_moe_layer_e4m3(const hb_w3_experts* routed, const hb_w3_experts* shared, const float* gate_vec, const void* x,
                                    const int32_t* ids, const float* weights, int m, int topk, void* out, void* workspace,
                                    size_t workspace_bytes, void* stream) {
  return moe_layer(routed, shared, gate_vec, x, ids, weights, m, topk, out, workspace, workspace_bytes, stream, 0, nullptr, true);
}

// ------------------------------------------------------------------------------- the entry point that allocates nothing
// hb_w3_moe_layer with its workspace in a device array of this library instead of a caller's buffer, for callers that
// cannot allocate. Every GPU the library runs on holds its own copy of the array at its own address; the array's name
// is a host-side stand-in, so the address is asked for once a device (hipGetSymbolAddress, with that device current)
// and only that pointer is ever handed to a kernel.
static __device__ __align__(256) uint8_t scratch[HB_STATIC_SCRATCH_BYTES];

namespace {
constexpr int SCRATCH_MAX_DEVICES = 64;
std::mutex g_scratch_lock;
void* g_scratch_ptr[SCRATCH_MAX_DEVICES] = {};

// The current device's copy of `scratch`, or null if the runtime will not say where it is.
void* scratch_of_current_device() {
  int device = -1;
  if (hipGetDevice(&device) != hipSuccess || device < 0 || device >= SCRATCH_MAX_DEVICES) return nullptr;
  std::lock_guard<std::mutex> hold(g_scratch_lock);
  if (!g_scratch_ptr[device]) {
    void* ptr = nullptr;
    if (hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)) != hipSuccess) return nullptr;
    g_scratch_ptr[device] = ptr;
  }
  return g_scratch_ptr[device];
}
}  // namespace

extern "C" int hb_w3_moe_layer_static(const hb_w3_experts* routed, const hb_w3_experts* shared, const float* gate_vec, const void* x,
                                      const int32_t* ids, const float* weights, int m, int topk, void* out, void* stream) {
  if (int e = check_experts(routed)) return e;
  if (m <= 0 || topk <= 0) return HB_EINVAL;
  // sized before anything is touched: the same carve as hb_w3_moe_workspace_bytes
  if (moe_carve(nullptr, m, topk, routed->experts, routed->inter, routed->hidden_out, shared ? 1 : 0, routed->hidden).bytes > HB_STATIC_SCRATCH_BYTES)
    return HB_ESCRATCH;
  void* ptr = scratch_of_current_device();
  if (!ptr) return HB_ELAUNCH;
  return moe_layer(routed, shared, gate_vec, x, ids, weights, m, topk, out, ptr, HB_STATIC_SCRATCH_BYTES, stream, 0, nullptr);
}

// ------------------------------------------------------------------------------------- a workspace's head words
__global__ __launch_bounds__(256) void workspace_zero_kernel(uint32_t* at, size_t words) {
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < words; i += (size_t)gridDim.x * 256) at[i] = 0u;
}

extern "C" int hb_workspace_reset(void* workspace, size_t workspace_bytes, void* stream) {
  if (!workspace) {  // the library's own scratch (hb_w3_moe_layer_static)
    workspace = scratch_of_current_device();
    workspace_bytes = HB_STATIC_SCRATCH_BYTES;
    if (!workspace) return HB_ELAUNCH;
  }
  if (!aligned(workspace, 16) || workspace_bytes < 4) return HB_EINVAL;
  const size_t words = std::min<size_t>(workspace_bytes, HB_WORKSPACE_ZERO_BYTES) / 4;
  hipLaunchKernelGGL(workspace_zero_kernel, dim3((unsigned)std::min<size_t>((words + 255) / 256, 1024)), dim3(256), 0, as_stream(stream),
                     static_cast<uint32_t*>(workspace), words);
  return launch_status();
}

extern "C" int hb_workspace_status(const void* workspace, int32_t* status, int wait, void* stream) {
  if (!status) return HB_ENULL;
  if (!workspace) workspace = scratch_of_current_device();
  if (!workspace) return HB_ELAUNCH;
  if (!aligned(workspace, 16)) return HB_EINVAL;
  if (hipMemcpyAsync(status, static_cast<const int32_t*>(workspace) + PLAN_FAULT, sizeof(int32_t), hipMemcpyDeviceToHost, as_stream(stream)) != hipSuccess)
    return HB_ELAUNCH;
  if (wait && hipStreamSynchronize(as_stream(stream)) != hipSuccess) return HB_ELAUNCH;
  return HB_OK;
}

extern "C" int hb_w3_moe_layer_logits(const hb_w3_experts* routed, const hb_w3_experts* shared, const float* gate_vec, const void* x,
                                      const float* logits, int experts_total, int m, int topk, int32_t* ids, float* weights, void* out,
                                      void* workspace, size_t workspace_bytes, void* stream) {
  if (!logits) return HB_ENULL;
  if (!aligned(logits, 4)) return HB_EINVAL;
  const Routing route{{logits, 0, experts_total, nullptr, 1}, ids, weights};
  return moe_layer(routed, shared, gate_vec, x, ids, weights, m, topk, out, workspace, workspace_bytes, stream, experts_total, &route);
}

extern "C" int hb_w3_moe_layer_budget(const hb_w3_experts* routed, const hb_w3_experts* shared, const float* gate_vec, const void* x,
                                      const void* logits, int experts_total, int m, int topk, int keep, int budget, const int32_t* slots, int steps,
                                      int per_request, int min_cap, int32_t* ids, float* weights, void* out, void* workspace,
                                      size_t workspace_bytes, void* stream) {
  if (!logits) return HB_ENULL;
  const BudgetRoute b{static_cast<const uint16_t*>(logits), experts_total, keep, budget, steps, 0, per_request, min_cap, slots};
  const Routing route{{}, ids, weights, &b};
  return moe_layer(routed, shared, gate_vec, x, ids, weights, m, topk, out, workspace, workspace_bytes, stream, experts_total, &route);
}

extern "C" int hb_w3_moe_layer_logits_e4m3(const hb_w3_experts* routed, const hb_w3_experts* shared, const float* gate_vec, const void* x,
                                           const float* logits, int experts_total, int m, int topk, int32_t* ids, float* weights, void* out,
                                           void* workspace, size_t workspace_bytes, void* stream) {
  if (!logits) return HB_ENULL;
  if (!aligned(logits, 4)) return HB_EINVAL;
  const Routing route{{logits, 0, experts_total, nullptr, 1}, ids, weights};
  return moe_layer(routed, shared, gate_vec, x, ids, weights, m, topk, out, workspace, workspace_bytes, stream, experts_total, &route, true);
}

// The layer from its input rows: [workspace of the routed call][BF16 logits, where the call makes them][ids][weights].
namespace {
struct LayerScratch {
  size_t moe;  // the routed call's bytes
  uint16_t* logits;
  int32_t* ids;
  float* weights;
  size_t bytes;
};
LayerScratch layer_scratch(void* base, size_t moe, int m, int topk, int experts_total) {
  LayerScratch l{moe, nullptr, nullptr, nullptr, 0};
  size_t off = moe;
  auto take = [&](size_t bytes) {
    void* ptr = base ? static_cast<char*>(base) + off : nullptr;
    off += (bytes + 255) & ~(size_t)255;
    return ptr;
  };
  l.logits = static_cast<uint16_t*>(take(m <= MOE_ROUTER_ROWS ? (size_t)m * experts_total * 2 : 0));
  l.ids = static_cast<int32_t*>(take((size_t)m * topk * 4));
  l.weights = static_cast<float*>(take((size_t)m * topk * 4));
  l.bytes = off;
  return l;
}
}  // namespace

extern "C" size_t hb_w3_moe_layer_rows_workspace_bytes(int m, int topk, const hb_w3_experts* routed, int shared, int experts_total) {
  const size_t moe = hb_w3_moe_workspace_bytes(m, topk, routed, shared);
  return moe && experts_total > 0 ? layer_scratch(nullptr, moe, m, topk, experts_total).bytes : 0;
}

extern "C" int hb_w3_moe_layer_rows(const hb_w3_experts* routed, const hb_w3_experts* shared, const float* gate_vec, const void* x, const void* router,
                                    const void* logits, int experts_total, int m, int topk, int keep, int budget, const int32_t* slots, int steps,
                                    int per_request, int min_cap, void* out, void* workspace, size_t workspace_bytes, void* stream) {
  if (int e = check_experts(routed)) return e;
  if (!x || !workspace || (!router && !logits)) return HB_ENULL;
  if (m <= 0 || topk <= 0 || experts_total <= 0 || steps <= 0) return HB_EINVAL;
  if (!aligned(x, 16) || (!logits && !aligned(router, 16)) || !aligned(logits, 2) || !aligned(slots, 4) || !aligned(workspace, 16)) return HB_EINVAL;
  if (!logits && m > MOE_ROUTER_ROWS) return HB_EINVAL;
  const size_t moe = hb_w3_moe_workspace_bytes(m, topk, routed, shared != nullptr);
  const LayerScratch l = layer_scratch(workspace, moe, m, topk, experts_total);
  if (!moe || workspace_bytes < l.bytes) return HB_EWORKSPACE;
  const uint16_t* lg = static_cast<const uint16_t*>(logits);
  if (!lg) {
    moe_launch_router(static_cast<const uint16_t*>(x), static_cast<const uint16_t*>(router), m, experts_total, routed->hidden, l.logits, as_stream(stream));
    lg = l.logits;
  }
  const BudgetRoute b{lg, experts_total, keep, budget, steps, 0, per_request, min_cap, slots};
  const Routing route{{lg, 1, experts_total, slots, steps}, l.ids, l.weights, budget > 0 ? &b : nullptr};
  return moe_layer(routed, shared, gate_vec, x, l.ids, l.weights, m, topk, out, workspace, l.moe, stream, experts_total, &route);
}
