// NVFP4 (E2M1 codes, E4M3 scale per 16 weights, FP32 global scale) weight-only kernels for gfx950.
//
// Tile layout: blocks of 64 output rows x 128 k, NVFP4_BLOCK_BYTES each, [rows/64][K/128]:
//   bytes    0..4095  codes: four 128-bit loads per lane, load nt of lane l at (nt * 64 + l) * 16. Lane l = 16 q + r owns,
//                     for the 16-row tile nt, the weights of row 64 nb + 16 nt + r: dword s holds k = 128 c + 32 s + 8 q .. + 7,
//                     nibble i the i-th. That is the lane's operand of v_mfma_f32_16x16x32_bf16 for the 32-k step s, eight
//                     consecutive k of ONE 16-block (2 s + q / 2), so the activations' side is one 16-byte piece of a row
//                     and an expansion has one block scale.
//   bytes 4096..4607  scales: 16 B per row-in-tile r and block parity u at 4096 + 16 (2 r + u): byte 4 nt + s is the E4M3
//                     scale of row 64 nb + 16 nt + r, block 8 c + 2 s + u - the sixteen scales of lane (q, r), u = q / 2.
// Codes expand with v_cvt_scalef32_pk_{bf16,f32}_fp4 (two weights per instruction, exact).
#include <string.h>

#include <atomic>
#include <cmath>

#include "panel_kernel.hpp"
#include "plan.hpp"
#include "ring.hpp"
#include "stream_common.hpp"

namespace hb {

constexpr int NVFP4_BLOCK_BYTES = 4608;
constexpr int NVFP4_SCALE_OFFSET = 4096;
typedef __attribute__((ext_vector_type(2))) uint32_t u32x2_t;

__host__ __device__ inline int64_t swizzled_scale_offset(int64_t r, int c, int groups_pad) {
  return (r / 128) * 128 * groups_pad + (c / 4) * 512 + (r % 32) * 16 + ((r / 32) % 4) * 4 + c % 4;
}

// One thread per (block, tile, lane): the lane's four code dwords of one 16-row tile.
__global__ __launch_bounds__(256) void nvfp4_repack_codes_kernel(const uint8_t* __restrict__ weight, int64_t blocks, int chunks,
                                                                 uint8_t* __restrict__ tiled) {
  const int64_t id = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (id >= blocks * 256) return;
  const int64_t blk = id >> 8;
  const int nt = (int)(id >> 6) & 3, lane = (int)(id & 63), q = lane >> 4, r = lane & 15;
  const int64_t nb = blk / chunks;
  const int c = (int)(blk % chunks);
  const int64_t n = nb * 64 + nt * 16 + r;
  const uint8_t* src = weight + n * (chunks * 64) + c * 64 + 4 * q;  // 64 bytes per chunk per row, 16 a step
  uint32_t d[4];
#pragma unroll
  for (int e = 0; e < 4; e++) d[e] = src[16 * e] | (uint32_t)src[16 * e + 1] << 8 | (uint32_t)src[16 * e + 2] << 16 | (uint32_t)src[16 * e + 3] << 24;
  *reinterpret_cast<u32x4_t*>(tiled + blk * NVFP4_BLOCK_BYTES + (nt * 64 + lane) * 16) = u32x4_t{d[0], d[1], d[2], d[3]};
}

// One thread per scale byte.
__global__ __launch_bounds__(256) void nvfp4_repack_scales_kernel(const uint8_t* __restrict__ scales, int swizzled, int64_t blocks,
                                                                  int chunks, uint8_t* __restrict__ tiled) {
  const int64_t id = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (id >= blocks * 512) return;
  const int64_t blk = id >> 9;
  const int within = (int)(id & 511), r = within >> 5, u = (within >> 4) & 1, nt = (within >> 2) & 3, b = 2 * (within & 3) + u;
  const int64_t nb = blk / chunks;
  const int c = (int)(blk % chunks);
  const int64_t n = nb * 64 + nt * 16 + r;
  const int groups = chunks * 8, g = 8 * c + b;
  const uint8_t v = swizzled ? scales[swizzled_scale_offset(n, g, (groups + 3) / 4 * 4)] : scales[n * groups + g];
  tiled[blk * NVFP4_BLOCK_BYTES + NVFP4_SCALE_OFFSET + within] = v;
}

__device__ __forceinline__ float e2m1_to_f32(uint32_t code) {
  const uint32_t a = code & 7u;
  const float mag = a < 4u ? 0.5f * (float)a : a == 4u ? 2.0f : a == 5u ? 3.0f : a == 6u ? 4.0f : 6.0f;
  return (code & 8u) ? -mag : mag;
}

// One thread per (block, tile, lane): 32 dequantized weights, e2m1 * float(scale) then * global (two roundings).
__global__ __launch_bounds__(256) void nvfp4_dequant_kernel(const uint8_t* __restrict__ tiled, float global_scale, int64_t blocks, int chunks,
                                                            float* __restrict__ out) {
  const int64_t id = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (id >= blocks * 256) return;
  const int64_t blk = id >> 8;
  const int nt = (int)(id >> 6) & 3, lane = (int)(id & 63), q = lane >> 4, r = lane & 15;
  const int64_t nb = blk / chunks;
  const int c = (int)(blk % chunks);
  const int k = chunks * 128;
  const uint8_t* base = tiled + blk * NVFP4_BLOCK_BYTES;
  const int64_t n = nb * 64 + nt * 16 + r;
  const u32x4_t d = *reinterpret_cast<const u32x4_t*>(base + (nt * 64 + lane) * 16);
  const uint32_t dw[4] = {d.x, d.y, d.z, d.w};
  for (int t = 0; t < 4; t++) {
    const float s = e4m3_to_f32(base[NVFP4_SCALE_OFFSET + 16 * (2 * r + (q >> 1)) + 4 * nt + t]);
    float* o = out + n * k + c * 128 + 32 * t + 8 * q;
#pragma unroll
    for (int i = 0; i < 8; i++) o[i] = __fmul_rn(__fmul_rn(e2m1_to_f32((dw[t] >> (4 * i)) & 15u), s), global_scale);
  }
}

struct Fp4Chunk {  // the weight side of a chunk: four 16-row tiles of codes (a dword a step), their block scales (a dword a tile, a byte a step)
  u32x4_t w0, w1, w2, w3, sc;
  __device__ __forceinline__ const u32x4_t& tile(int nt) const { return nt == 0 ? w0 : nt == 1 ? w1 : nt == 2 ? w2 : w3; }
};

// Byte S of a dword of E4M3 scales as FP32.
template <int S>
__device__ __forceinline__ float fp4_scale(uint32_t sc) { return __builtin_amdgcn_cvt_f32_fp8(sc, S); }

// The eight weights of one code dword as they are (the block scale is folded into the sums) ...
__device__ __forceinline__ bf16x8_t fp4_plain(uint32_t codes) {
  u32x4_t b;
  b.x = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(codes, 1.0f, 0));
  b.y = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(codes, 1.0f, 1));
  b.z = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(codes, 1.0f, 2));
  b.w = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(codes, 1.0f, 3));
  return __builtin_bit_cast(bf16x8_t, b);
}
// ... and times their block's scale: a product of a 2-bit and a 4-bit significand, exact in BF16.
__device__ __forceinline__ bf16x8_t fp4_scaled(uint32_t codes, float s) {
  const f32x2_pair_t a = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(codes, 1.0f, 0), b = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(codes, 1.0f, 1);
  const f32x2_pair_t c = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(codes, 1.0f, 2), d = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(codes, 1.0f, 3);
  return __builtin_bit_cast(bf16x8_t, u32x4_t{bf16_pair(a.x * s, a.y * s), bf16_pair(b.x * s, b.y * s), bf16_pair(c.x * s, c.y * s), bf16_pair(d.x * s, d.y * s)});
}

__device__ __forceinline__ f32x4_t fp4_mfma(const u32x4_t& a, const bf16x8_t& b, const f32x4_t& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), b, c, 0, 0, 0);
}
__device__ __forceinline__ void fp4_fold(const f32x4_t& part, float s, f32x4_t& acc) {
  acc.x = fmaf(part.x, s, acc.x);
  acc.y = fmaf(part.y, s, acc.y);
  acc.z = fmaf(part.z, s, acc.z);
  acc.w = fmaf(part.w, s, acc.w);
}

// ------------------------------------------------------------------------------------------------ the weight ring
// (ring.hpp) for NVFP4 blocks: four 16-byte loads a lane of codes, two 4-byte loads a lane of scales. U: the bit of q that
// names the parity of the blocks whose scales the lane reads (1: its own weights' blocks; 0: see Fp4Few4Acts).
template <int U>
struct Fp4RingOf {
  typedef Fp4Chunk Chunk;
  static constexpr int BLOCK_BYTES = NVFP4_BLOCK_BYTES, LOADS = 6;
  static __device__ __forceinline__ void lanes(RingSource& src, int lane, int r16, uint32_t slot0, uint32_t& codes, uint32_t& scales) {
    src.codes = 16u * lane;
    src.scales = 4u * lane;
    codes = slot0 + 16u * lane;
    scales = slot0 + 32u * r16 + 16u * ((lane >> (4 + U)) & 1);
  }
  static __device__ __forceinline__ void request(const RingSource& src, int chunk, lds_ptr_t slot) {
    const uint32_t at = (uint32_t)chunk * NVFP4_BLOCK_BYTES;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(src.row, slot, 16, src.codes, at, 0, 2);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(src.row, slot, 16, src.codes, at, 1024, 2);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(src.row, slot, 16, src.codes, at, 2048, 2);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(src.row, slot, 16, src.codes, at, 3072, 2);
    // the instruction's offset field (which moves both ends) stops at 4095: the scales' place is given by hand
    __builtin_amdgcn_raw_ptr_buffer_load_lds(src.row, slot + NVFP4_SCALE_OFFSET, 4, src.scales, at + NVFP4_SCALE_OFFSET, 0, 2);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(src.row, slot + NVFP4_SCALE_OFFSET, 4, src.scales, at + NVFP4_SCALE_OFFSET, 256, 2);
    __builtin_amdgcn_sched_barrier(0);  // asked for here, not wherever the scheduler would sink it below the arithmetic
  }
  // the reads of a block from slot 0, and (after a wait) their values
  static __device__ __forceinline__ void ask(Chunk& ch, uint32_t codes, uint32_t scales) {
    ask_lds<0>(ch.w0, codes);
    ask_lds<1024>(ch.w1, codes);
    ask_lds<2048>(ch.w2, codes);
    ask_lds<3072>(ch.w3, codes);
    ask_lds<NVFP4_SCALE_OFFSET>(ch.sc, scales);
  }
  static __device__ __forceinline__ void have(Chunk& ch) {
    pin(ch.w0);
    pin(ch.w1);
    pin(ch.w2);
    pin(ch.w3);
    pin(ch.sc);
  }
  template <int BEHIND, int SLOT>
  static __device__ __forceinline__ void take(Chunk& ch, uint32_t codes, uint32_t scales) {
    asm volatile(
        "s_waitcnt vmcnt(%7)\n\t"
        "ds_read_b128 %0, %5 offset:%8\n\t"
        "ds_read_b128 %1, %5 offset:%9\n\t"
        "ds_read_b128 %2, %5 offset:%10\n\t"
        "ds_read_b128 %3, %5 offset:%11\n\t"
        "ds_read_b128 %4, %6 offset:%12\n\t"
        "s_waitcnt lgkmcnt(0)"  // the slot is read: it may be given to another chunk
        : "=&v"(ch.w0), "=&v"(ch.w1), "=&v"(ch.w2), "=&v"(ch.w3), "=&v"(ch.sc)
        : "v"(codes), "v"(scales), "n"(BEHIND), "n"(SLOT * NVFP4_BLOCK_BYTES), "n"(SLOT * NVFP4_BLOCK_BYTES + 1024), "n"(SLOT * NVFP4_BLOCK_BYTES + 2048),
          "n"(SLOT * NVFP4_BLOCK_BYTES + 3072), "n"(SLOT * NVFP4_BLOCK_BYTES + NVFP4_SCALE_OFFSET)
        : "memory");
  }
};
typedef Fp4RingOf<1> Fp4Ring;
// A ring that brings in only the codes of the 16-row tiles T0 .. T1 - 1 (a load a tile) and the scales. The Chunk's other
// registers stay unset and unread.
template <int U, int T0, int T1>
struct Fp4RingPart : Fp4RingOf<U> {
  typedef Fp4Chunk Chunk;
  static constexpr int TILES = T1 - T0, LOADS = TILES + 2;
  static_assert(0 <= T0 && T1 <= 4 && (TILES == 1 || TILES == 2), "a tile or a pair of tiles");
  static __device__ __forceinline__ void request(const RingSource& src, int chunk, lds_ptr_t slot) {
    const uint32_t at = (uint32_t)chunk * NVFP4_BLOCK_BYTES;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(src.row, slot, 16, src.codes, at, 1024 * T0, 2);
    if (TILES == 2) __builtin_amdgcn_raw_ptr_buffer_load_lds(src.row, slot, 16, src.codes, at, 1024 * (T1 - 1), 2);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(src.row, slot + NVFP4_SCALE_OFFSET, 4, src.scales, at + NVFP4_SCALE_OFFSET, 0, 2);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(src.row, slot + NVFP4_SCALE_OFFSET, 4, src.scales, at + NVFP4_SCALE_OFFSET, 256, 2);
    __builtin_amdgcn_sched_barrier(0);
  }
  static __device__ __forceinline__ u32x4_t& load_of(Chunk& ch, int t) { return t == 0 ? ch.w0 : t == 1 ? ch.w1 : t == 2 ? ch.w2 : ch.w3; }
  template <int BEHIND, int SLOT>
  static __device__ __forceinline__ void take(Chunk& ch, uint32_t codes, uint32_t scales) {
    if (TILES == 2) {
      asm volatile(
          "s_waitcnt vmcnt(%5)\n\t"
          "ds_read_b128 %0, %3 offset:%6\n\t"
          "ds_read_b128 %1, %3 offset:%7\n\t"
          "ds_read_b128 %2, %4 offset:%8\n\t"
          "s_waitcnt lgkmcnt(0)"
          : "=&v"(load_of(ch, T0)), "=&v"(load_of(ch, T1 - 1)), "=&v"(ch.sc)
          : "v"(codes), "v"(scales), "n"(BEHIND), "n"(SLOT * NVFP4_BLOCK_BYTES + 1024 * T0), "n"(SLOT * NVFP4_BLOCK_BYTES + 1024 * (T1 - 1)),
            "n"(SLOT * NVFP4_BLOCK_BYTES + NVFP4_SCALE_OFFSET)
          : "memory");
    } else {
      asm volatile(
          "s_waitcnt vmcnt(%4)\n\t"
          "ds_read_b128 %0, %2 offset:%5\n\t"
          "ds_read_b128 %1, %3 offset:%6\n\t"
          "s_waitcnt lgkmcnt(0)"
          : "=&v"(load_of(ch, T0)), "=&v"(ch.sc)
          : "v"(codes), "v"(scales), "n"(BEHIND), "n"(SLOT * NVFP4_BLOCK_BYTES + 1024 * T0), "n"(SLOT * NVFP4_BLOCK_BYTES + NVFP4_SCALE_OFFSET)
          : "memory");
    }
  }
};
constexpr int FP4_RING_BYTES = ring_bytes<Fp4Ring>();  // LDS per wavefront; its first 4 KB double as the K-split exchange

// ---------------------------------------------------------------------------------------- slots of one to eight rows
//
// With few rows in the slot the sixteen MFMA rows carry several 16-blocks at once, so that a block scale is folded into
// the sums of many weights' products instead of being multiplied into every weight, and the activations are one or two
// 16-byte loads a lane and chunk.
//
// Up to eight rows: A row 8 u + i holds row i of the slot over the lanes of block parity u only (q / 2 == u; zero over
// the others), so step s leaves block 2 s + u's partial sums in its output rows 8 u .. 8 u + 7: lane (q, r16) ends up with
// parity q / 2 of slot rows 4 (q % 2) .. + 3 - the parity of its own weights' scales. Sixteen scale conversions and 64
// multiply-adds a chunk.
//
// Up to four rows: two steps 2 t, 2 t + 1 chain into one result. A row 4 j + i holds row i over the blocks 4 t + j only:
// step 2 t + j / 2 and the lanes of parity j % 2. Lane (q, r16) ends up with block 4 t + q of the slot's four rows: its
// scale is the byte 2 t + q / 2 of parity q % 2 (the ring hands the lane that parity's). Eight conversions and 32
// multiply-adds a chunk.
//
// The blocks' sums are added across the lanes after the last chunk, which leaves the sixteen-row layout.
constexpr int FP4_FEW_ROWS = 8, FP4_FEWER_ROWS = 4;

// What a lane reads whose weights are not of its A row's parity: zeros, from here. That spares sixteen selects a chunk and
// half of the activations' way through the L1 (eight rows, 25600 x 5120: 17.1 us, with the selects 19.3).
__device__ const u32x4_t fp4_zero_piece[16] = {};

template <int T0 = 0, int T1 = 4>  // the 16-row tiles T0 .. T1 - 1 of the block (the other accumulators stay zero)
struct Fp4Few8Acts {
  static constexpr int LOADS = 4;
  u32x4_t even[4], odd[4];  // the lane's piece of each step of the next even and the next odd chunk
  const uint16_t* at;       // the lane's piece of step 0 of the wavefront's first chunk ...
  uint32_t stride;          // ... and the elements to the next chunk's (0: the zeros)
  __device__ __forceinline__ void load(u32x4_t (&to)[4], int i) const {
    const uint16_t* from = at + i * stride;
#pragma unroll
    for (int s = 0; s < 4; s++) to[s] = *(const __attribute__((address_space(1))) u32x4_t*)(from + 32 * s);  // (said to be global: the compiler cannot tell of the two)
  }
  template <int EPI>
  __device__ __forceinline__ void start(const StreamParams& p, const Slot& sl, int, int c0, int n, int lane) {
    const int q = lane >> 4, r16 = lane & 15;
    const bool mine = (r16 >> 3) == (q >> 1);
    at = mine ? activation_row<EPI>(p, sl, r16 & 7) + (int64_t)c0 * 128 + 8 * q : reinterpret_cast<const uint16_t*>(fp4_zero_piece);
    stride = mine ? 128 : 0;
    load(even, 0);
    if (n > 1) load(odd, 1);
  }
  template <int S>
  __device__ __forceinline__ void one(uint32_t codes, uint32_t sc, const u32x4_t& a, f32x4_t& acc) const {
    fp4_fold(fp4_mfma(a, fp4_plain(codes), f32x4_t{0.f, 0.f, 0.f, 0.f}), fp4_scale<S>(sc), acc);
  }
  __device__ __forceinline__ void tile(const u32x4_t& w, uint32_t sc, const u32x4_t (&a)[4], f32x4_t& acc) const {
    one<0>(w.x, sc, a[0], acc);
    one<1>(w.y, sc, a[1], acc);
    one<2>(w.z, sc, a[2], acc);
    one<3>(w.w, sc, a[3], acc);
  }
  template <int ODD, bool MORE2, bool MORE1>
  __device__ __forceinline__ void step(const Fp4Chunk& ch, int i, f32x4_t& acc0, f32x4_t& acc1, f32x4_t& acc2, f32x4_t& acc3, const Slot&) {
    const u32x4_t(&a)[4] = ODD ? odd : even;
    if (T0 <= 0 && 0 < T1) tile(ch.w0, ch.sc.x, a, acc0);
    __builtin_amdgcn_sched_barrier(0);  // a tile at a time: interleaving the four costs more registers than there are
    if (T0 <= 1 && 1 < T1) tile(ch.w1, ch.sc.y, a, acc1);
    __builtin_amdgcn_sched_barrier(0);
    if (T0 <= 2 && 2 < T1) tile(ch.w2, ch.sc.z, a, acc2);
    __builtin_amdgcn_sched_barrier(0);
    if (T0 <= 3 && 3 < T1) tile(ch.w3, ch.sc.w, a, acc3);
    if (MORE2) {
      if (ODD) load(odd, i + 2); else load(even, i + 2);
    }
  }
};

template <int T0 = 0, int T1 = 4>
struct Fp4Few4Acts {
  static constexpr int LOADS = 2;
  u32x4_t even[2], odd[2];  // the lane's piece of the pairs of steps of the next even and the next odd chunk
  bool first, second;       // the step of a pair this lane's A row takes its block from (neither: the block's other lanes)
  uint32_t shift;           // 8 * (q / 2)
  const uint16_t* at;       // the lane's piece of pair 0 of the wavefront's first chunk
  __device__ __forceinline__ void load(u32x4_t (&to)[2], int i) const {
    to[0] = *reinterpret_cast<const u32x4_t*>(at + (int64_t)i * 128);
    to[1] = *reinterpret_cast<const u32x4_t*>(at + (int64_t)i * 128 + 64);
  }
  template <int EPI>
  __device__ __forceinline__ void start(const StreamParams& p, const Slot& sl, int, int c0, int n, int lane) {
    const int q = lane >> 4, r16 = lane & 15, j = r16 >> 2;
    const bool mine = (j & 1) == (q >> 1);
    first = mine && j < 2;
    second = mine && j >= 2;
    shift = 8 * (q >> 1);
    at = activation_row<EPI>(p, sl, r16 & 3) + (int64_t)c0 * 128 + 32 * (j >> 1) + 8 * q;
    load(even, 0);
    if (n > 1) load(odd, 1);
  }
  static __device__ __forceinline__ u32x4_t masked(const u32x4_t& v, bool keep) { return u32x4_t{keep ? v.x : 0u, keep ? v.y : 0u, keep ? v.z : 0u, keep ? v.w : 0u}; }
  __device__ __forceinline__ void tile(const u32x4_t& w, uint32_t sc, const u32x4_t (&a)[4], f32x4_t& acc) const {
    const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
    const uint32_t mine = sc >> shift;
    fp4_fold(fp4_mfma(a[1], fp4_plain(w.y), fp4_mfma(a[0], fp4_plain(w.x), zero)), fp4_scale<0>(mine), acc);
    fp4_fold(fp4_mfma(a[3], fp4_plain(w.w), fp4_mfma(a[2], fp4_plain(w.z), zero)), fp4_scale<2>(mine), acc);
  }
  template <int ODD, bool MORE2, bool MORE1>
  __device__ __forceinline__ void step(const Fp4Chunk& ch, int i, f32x4_t& acc0, f32x4_t& acc1, f32x4_t& acc2, f32x4_t& acc3, const Slot&) {
    u32x4_t a[4];
#pragma unroll
    for (int t = 0; t < 2; t++) {
      a[2 * t] = masked(ODD ? odd[t] : even[t], first);
      a[2 * t + 1] = masked(ODD ? odd[t] : even[t], second);
    }
    if (T0 <= 0 && 0 < T1) tile(ch.w0, ch.sc.x, a, acc0);
    if (T0 <= 1 && 1 < T1) tile(ch.w1, ch.sc.y, a, acc1);
    if (T0 <= 2 && 2 < T1) tile(ch.w2, ch.sc.z, a, acc2);
    if (T0 <= 3 && 3 < T1) tile(ch.w3, ch.sc.w, a, acc3);
    if (MORE2) {
      if (ODD) load(odd, i + 2); else load(even, i + 2);
    }
  }
};

__device__ __forceinline__ void add_lanes(f32x4_t& acc, int distance) {
  acc.x += __shfl_xor(acc.x, distance);
  acc.y += __shfl_xor(acc.y, distance);
  acc.z += __shfl_xor(acc.z, distance);
  acc.w += __shfl_xor(acc.w, distance);
}

// ------------------------------------------------------------------------------------------------ slots of more rows
//
// Nine to sixteen rows: every weight is expanded with its block scale multiplied in. Lane (q, r16) feeds row r16, k 8 q ..
// + 7 of a step: a chunk's four pieces rest in registers, and each is asked for again, for the next chunk, as soon as its
// products are issued - straight from the L2: a wavefront shares them with nobody and meets no barrier. The requests of a
// wavefront come back in order, so the next weights are asked for BEHIND those pieces (a piece that waited behind weights
// from memory would wait for them too): a block is on its way for the whole of the chunk before it.
//
// The body serves matrices past 4 GiB too, which the panel kernel does not take: a lane's 32-bit byte offset counts from the
// slot's first row (a uniform base: 2048 x 2048 at nine rows 8.6 us against 9.0 with a pointer a lane), and where the
// slot's rows are gathered, which may lie anywhere, the lane holds a whole pointer.
template <int EPI, int T0 = 0, int T1 = 4, class Ring = Fp4Ring>  // the 16-row tiles T0 .. T1 - 1 of the block
struct Fp4Full {
  static constexpr int TILES = T1 - T0;
  f32x4_t acc[4];
  u32x4_t a[4];
  const uint8_t* x;  // step 0 of the wavefront's first chunk: of the slot's first row (the same for all lanes) or, gathered, the lane's own piece ...
  uint32_t at;       // ... and from there to the lane's piece
  __device__ __forceinline__ u32x4_t piece(int i, int s) const { return *reinterpret_cast<const u32x4_t*>(x + (size_t)i * 256 + 64 * s + at); }
  __device__ __forceinline__ void start(const StreamParams& p, const Slot& sl, int c0, int lane) {
    const int r16 = lane & 15;
    if constexpr (epi_gathers(EPI)) {
      x = reinterpret_cast<const uint8_t*>(activation_row<EPI>(p, sl, r16) + (int64_t)c0 * 128 + 8 * (lane >> 4));
      at = 0;
    } else {
      x = reinterpret_cast<const uint8_t*>(p.a + (int64_t)sl.p0 * p.a_stride + (int64_t)c0 * 128);
      at = (uint32_t)(min(r16, sl.rows - 1) * p.a_stride) * 2 + 16 * (lane >> 4);
    }
#pragma unroll
    for (int nt = 0; nt < 4; nt++) acc[nt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < 4; s++) a[s] = piece(0, s);
  }
  template <int J>  // fragment J = TILES * step + tile - T0 of a chunk
  static __device__ __forceinline__ bf16x8_t fragment(const Fp4Chunk& ch) {
    constexpr int S = J / TILES, NT = T0 + J % TILES;
    return fp4_scaled(ch.tile(NT)[S], fp4_scale<S>(ch.sc[NT]));
  }
  // The product of fragment J, and behind it the expansion of the next fragment: a product holds the matrix core for
  // sixteen cycles and the issue port for about seven of them.
  template <int J>
  __device__ __forceinline__ void fragments(const Fp4Chunk& ch, int i, bool more, bf16x8_t b) {
    if constexpr (J < 4 * TILES) {
      constexpr int S = J / TILES, NT = T0 + J % TILES;
      bf16x8_t next{};
      if constexpr (J + 1 < 4 * TILES) next = fragment<J + 1>(ch);
      acc[NT] = fp4_mfma(a[S], b, acc[NT]);
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x002, 17, 0);
      if (NT == T1 - 1) {
        u32x4_t held = __builtin_bit_cast(u32x4_t, next);
        asm volatile("" : "+v"(held));  // expanded here, beside the product, not behind the branch
        next = __builtin_bit_cast(bf16x8_t, held);
      }
      __builtin_amdgcn_sched_barrier(0);
      if (NT == T1 - 1 && more) a[S] = piece(i + 1, S);  // uniform
      fragments<J + 1>(ch, i, more, next);
    }
  }
  // One loop body for every chunk: the ring's slot by its parity, what is still to come by uniform branches.
  template <class Wait>
  __device__ __forceinline__ void run(const StreamParams& p, const Slot& sl, int nb, int c0, int c1, int lane, uint8_t* ring, Wait& wait) {
    const int n = c1 - c0;
    RingSource src;
    src.row = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(sl.w + (int64_t)nb * p.chunks * NVFP4_BLOCK_BYTES), 0, p.chunks * NVFP4_BLOCK_BYTES, 0x00020000);
    const lds_ptr_t slot0 = (lds_ptr_t)ring;
    uint32_t codes, scales;
    Ring::lanes(src, lane, lane & 15, (uint32_t)(uintptr_t)slot0, codes, scales);
    wait.look();
    Ring::request(src, c0, slot0);
    asm volatile("" ::: "memory");
    if constexpr (Wait::WAITS) {  // (the second block ahead of the first pieces, here: they are on their way together)
      if (n > 1) Ring::request(src, c0 + 1, slot0 + NVFP4_BLOCK_BYTES);
      if (!wait.done()) return;
    }
    start(p, sl, c0, lane);
    asm volatile("" ::: "memory");
    if (!Wait::WAITS && n > 1) Ring::request(src, c0 + 1, slot0 + NVFP4_BLOCK_BYTES);
    for (int i = 0; i < n; i++) {
      const uint32_t slot = (i & 1) * NVFP4_BLOCK_BYTES;
      Fp4Chunk ch;
      if (i + 1 < n) {
        Ring::template take<4 + Ring::LOADS, 0>(ch, codes + slot, scales + slot);
      } else {
        Ring::template take<4, 0>(ch, codes + slot, scales + slot);
      }
      fragments<0>(ch, i, i + 1 < n, fragment<0>(ch));
      if (i + 2 < n) Ring::request(src, c0 + i + 2, slot0 + slot);
    }
  }
};

// y = x Wq^T, dense or grouped by the expert plan: one wavefront per (64-row block, K range, slot of 16 activation rows),
// the same launch shape, slot table, weight ring, K-split exchange and epilogues as the W3 stream.
template <int EPI, class Wait>
__device__ __forceinline__ void nvfp4_workgroup(const StreamParams& p, int slot, int bx, uint8_t* rings, Wait& wait) {
  const Slot sl = slot_of<EPI>(p, slot);
  if (sl.rows <= 0) return;  // a slot the plan did not fill: the whole workgroup leaves
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // the same in every lane: kept in scalars
  if (wave >= p.ks * p.nbw) return;  // a launch shared with a matrix that takes more wavefronts a workgroup
  const WaveShare share = wave_share(p, wave);
  const int ks = share.ks, nbi = share.nbi, nb = bx * p.nbw + nbi;
  const bool active = nb < p.n_blocks;
  f32x4_t acc0 = {0.f, 0.f, 0.f, 0.f}, acc1 = acc0, acc2 = acc0, acc3 = acc0;
  if (active) {  // at least one chunk: the launch keeps ks <= chunks
    uint8_t* ring = rings + wave * FP4_RING_BYTES;
    if (sl.rows <= FP4_FEWER_ROWS && !p.no_few) {  // uniform over the workgroup
      stream_block_behind<EPI, Fp4Few4Acts<>, Fp4RingOf<0>>(p, sl, 0, nb, share.c0, share.c1, lane, ring, acc0, acc1, acc2, acc3, wait);
      for (int d = 16; d <= 32; d *= 2) {  // the four blocks' sums: lane q = 0 now holds the slot's rows as the epilogue expects them
        add_lanes(acc0, d);
        add_lanes(acc1, d);
        add_lanes(acc2, d);
        add_lanes(acc3, d);
      }
    } else if (sl.rows <= FP4_FEW_ROWS && !p.no_few) {
      stream_block_behind<EPI, Fp4Few8Acts<>, Fp4Ring>(p, sl, 0, nb, share.c0, share.c1, lane, ring, acc0, acc1, acc2, acc3, wait);
      add_lanes(acc0, 32);  // the two parities': lanes q = 0, 1 hold slot rows 0 .. 7
      add_lanes(acc1, 32);
      add_lanes(acc2, 32);
      add_lanes(acc3, 32);
    } else {
      Fp4Full<EPI> full;
      full.run(p, sl, nb, share.c0, share.c1, lane, ring, wait);
      acc0 = full.acc[0];
      acc1 = full.acc[1];
      acc2 = full.acc[2];
      acc3 = full.acc[3];
    }
  } else if (Wait::WAITS) {
    wait.done();
  }
  if (!wait.there) return;
  finish_block<EPI, false, FP4_RING_BYTES / 4>(p, sl, RowScales{}, nb, active, ks, nbi, reinterpret_cast<float*>(rings), acc0, acc1, acc2, acc3);
}

template <int EPI>
__device__ __forceinline__ void nvfp4_workgroup(const StreamParams& p, int slot, int bx, uint8_t* rings) {
  NoWait none;
  nvfp4_workgroup<EPI>(p, slot, bx, rings, none);
}

template <int EPI>
__global__ __launch_bounds__(1024) void nvfp4_stream_kernel(StreamParams p) {
  extern __shared__ __align__(16) uint8_t rings[];
  nvfp4_workgroup<EPI>(p, blockIdx.y, blockIdx.x, rings);
}

// A dense call of a few slots whose blocks are fewer than half the compute units: PARTS workgroups a 64-row block and slot, each
// its 4 / PARTS 16-row tiles and only those tiles' codes. The sums and their order are those of one workgroup with the same K split. What bounds the
// undivided launch is the expansion on a part of the device, and a small one the loads of a whole block ahead of the first product.
// Traced, one workgroup a block and so, us: one row 1024 x 1024 4.5 and 3.4, 4096 x 2048 5.9 and 4.4, 2048 x 5120 8.1 and 5.5, 8192 x
// 5120 9.0 and 7.0; eight rows 1024 x 4096 8.3 and 6.0, 8192 x 1024 5.5 and 4.4, 4096 x 5120 10.2 and 7.1; twelve rows, K split eight ways
// and sixteen, 2048 x 5120 13.3, 8.6 and 8.0, 8192 x 5120 14.2, 10.8 and 9.8; 33 rows 2048 x 5120 13.0, 10.2 and 9.5. In two up to 256 blocks it
// gained up to two rows only (12288 x 5120 four rows 10.2 and 11.2).
template <int EPI, int T0, int T1>
__device__ __forceinline__ void nvfp4_part_block(const StreamParams& p, const Slot& sl, int nb, const WaveShare& share, int lane, int wave, uint8_t* rings) {
  f32x4_t acc[4];
#pragma unroll
  for (int t = 0; t < 4; t++) acc[t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  uint8_t* ring = rings + wave * FP4_RING_BYTES;
  if (sl.rows <= FP4_FEWER_ROWS && !p.no_few) {  // uniform over the workgroup
    stream_block<EPI, Fp4Few4Acts<T0, T1>, Fp4RingPart<0, T0, T1>>(p, sl, 0, nb, share.c0, share.c1, lane, ring, acc[0], acc[1], acc[2], acc[3]);
    for (int d = 16; d <= 32; d *= 2)
#pragma unroll
      for (int t = T0; t < T1; t++) add_lanes(acc[t], d);
  } else if (sl.rows <= FP4_FEW_ROWS && !p.no_few) {
    stream_block<EPI, Fp4Few8Acts<T0, T1>, Fp4RingPart<1, T0, T1>>(p, sl, 0, nb, share.c0, share.c1, lane, ring, acc[0], acc[1], acc[2], acc[3]);
#pragma unroll
    for (int t = T0; t < T1; t++) add_lanes(acc[t], 32);
  } else {
    Fp4Full<EPI, T0, T1, Fp4RingPart<1, T0, T1>> full;
    NoWait none;
    full.run(p, sl, nb, share.c0, share.c1, lane, ring, none);
#pragma unroll
    for (int t = T0; t < T1; t++) acc[t] = full.acc[t];
  }
  // finish_block for these tiles: the splits' sums through LDS, added in split order, an accumulator register a split and turn
  constexpr int STRIDE = FP4_RING_BYTES / 4;
  float* first = reinterpret_cast<float*>(rings);
  float* mine = first + wave * STRIDE;
#pragma unroll
  for (int t = T0; t < T1; t++)
#pragma unroll
    for (int r = 0; r < 4; r++) mine[(t * 4 + r) * 64 + lane] = acc[t][r];
  __syncthreads();
  for (int idx = 4 * T0 + share.ks; idx < 4 * T1; idx += p.ks) {
    const int t = idx >> 2, r = idx & 3;
    if (r >= sl.rows) continue;
    float v = 0.f;
    for (int s = 0; s < p.ks; s++) v += first[s * STRIDE + idx * 64 + lane];
    emit<EPI, false>(p, sl, RowScales{}, nb, t, r, lane >> 4, lane & 15, v, 0.f);
  }
}
template <int EPI, int PARTS>
__global__ __launch_bounds__(1024) void nvfp4_part_kernel(StreamParams p) {
  extern __shared__ __align__(16) uint8_t rings[];
  const int die = blockIdx.x & 7, local = blockIdx.x >> 3, part = local % PARTS, nb = local / PARTS * 8 + die;  // a block's workgroups on one die
  if (nb >= p.n_blocks) return;
  const Slot sl = slot_of<EPI>(p, blockIdx.y);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const WaveShare share = wave_share(p, wave);
  if constexpr (PARTS == 2) {
    if (part == 0) nvfp4_part_block<EPI, 0, 2>(p, sl, nb, share, lane, wave, rings); else nvfp4_part_block<EPI, 2, 4>(p, sl, nb, share, lane, wave, rings);
  } else {
    if (part == 0) nvfp4_part_block<EPI, 0, 1>(p, sl, nb, share, lane, wave, rings);
    else if (part == 1) nvfp4_part_block<EPI, 1, 2>(p, sl, nb, share, lane, wave, rings);
    else if (part == 2) nvfp4_part_block<EPI, 2, 3>(p, sl, nb, share, lane, wave, rings);
    else nvfp4_part_block<EPI, 3, 4>(p, sl, nb, share, lane, wave, rings);
  }
}

// Two matrices of different geometry in one launch (the routed experts' layer beside the shared expert's, which reads
// other activations): the first `first` workgroups are (slot, block group) of the dense `b`, slot-major - every one of
// them has a whole K range to stream, so they start first - the rest of the planned `a`. Should the two shapes differ
// in wavefronts a workgroup, the smaller one's workgroups retire the wavefronts they do not use.
template <int EPI_A, int EPI_B>
__global__ __launch_bounds__(1024) void nvfp4_twin_kernel(StreamParams a, StreamParams b, int groups_a, int groups_b, int first) {
  extern __shared__ __align__(16) uint8_t rings[];
  int id = blockIdx.x;
  if (id < first) {
    const int slot = id / groups_b;
    nvfp4_workgroup<EPI_B>(b, slot, id - slot * groups_b, rings);
  } else {
    id -= first;
    const int slot = id / groups_a;
    nvfp4_workgroup<EPI_A>(a, slot, id - slot * groups_a, rings);
  }
}

// fc1 and fc2 of a routed call on the stream in one launch, as w3_fc12_kernel: the same order of the grid, the same counters and waits. `first`:
// the workgroups of a dense matrix beside them (a shared expert's down projection), which come ahead of all others and wait for nothing.
template <int EPI1>
__global__ __launch_bounds__(1024) void nvfp4_fc12_kernel(StreamParams p1, StreamParams p2, StreamParams b, int groups1, int groups2, int slots, int lag, int first) {
  extern __shared__ __align__(16) uint8_t rings[];
  __shared__ int outcome;
  const int id = blockIdx.x;
  if (id < first) {
    nvfp4_workgroup<EPI_DENSE>(b, 0, id, rings);
    return;
  }
  const Fc12Place at = fc12_place(id - first, groups1, groups2, slots, lag);
  if (p1.plan[PLAN_HEADER + 4 * at.slot + 2] <= 0) return;  // a slot without rows
  if (at.is_fc1) {
    nvfp4_workgroup<EPI1>(p1, at.slot, at.index, rings);
    fc12_arrive(p1, at.slot);
  } else {
    SlotWait wait(p2, at.slot, &outcome, false);
    nvfp4_workgroup<EPI_FC2>(p2, at.slot, at.index, rings, wait);
  }
}

// The product of a small latent block's router: at most sixteen rows, fused[m, n] = x [router; fc1_latent]^T in
// FP32, its latent columns also rounded to BF16 (hibana/kernels/csrc/nemotron_moe.cu:496-558 of the reference).
// The product is bound by how fast a compute unit brings its columns in, so a workgroup has eight of them only: the sixteen columns of a product's
// weight operand are eight weight rows over two parts of K. PACKED (up to eight rows): the sixteen activation rows are likewise eight
// over both parts, and of the result the two quarters where the parts agree are kept; else a product each. With the launches below, the
// block of 512 experts (1024, 2688) and a shared one of 5376, router and block in two calls of six launches and in one, us: one row 54.0 and 48.2, four 80.2
// and 72.5, eight 113.7 and 104.8, nine 127.5 and 125.6, sixteen 166.6 and 164.8; this product alone 7.7 and 5.6 of eight rows, 9.2 and 7.8 of sixteen (traced).
constexpr int FRONT_WAVES = 8, FRONT_COLUMNS = 8;
struct FrontGemv {
  const uint16_t* w;  // BF16 [n, k]
  const uint16_t* x;  // BF16 [m, k]
  float* fused;       // FP32 [m, n]
  uint16_t* lat;      // BF16 [m, n - e]
  int n, k, m, e;
};
template <bool PACKED>
__global__ __launch_bounds__(64 * FRONT_WAVES) void latent_front_kernel(FrontGemv g) {
  __shared__ float part[FRONT_WAVES * 256];
  const int n0 = blockIdx.x * FRONT_COLUMNS;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), q = lane >> 4, r16 = lane & 15, half = r16 >> 3;
  const int per_part = g.k / (2 * FRONT_WAVES), steps = per_part / 32, k0 = 2 * wave * per_part;  // k % 512 == 0
  const uint16_t* wat = g.w + (int64_t)min(n0 + (r16 & 7), g.n - 1) * g.k + k0 + half * per_part + 8 * q;
  const uint16_t* xat = g.x + (int64_t)min(PACKED ? r16 & 7 : r16, g.m - 1) * g.k + k0 + (PACKED ? half * per_part : 0) + 8 * q;
  f32x4_t lower = {0.f, 0.f, 0.f, 0.f}, upper = lower;
  constexpr int BATCH = 8;
  for (int s0 = 0; s0 < steps; s0 += BATCH) {
    u32x4_t b[BATCH], a[BATCH], a2[BATCH];
#pragma unroll
    for (int j = 0; j < BATCH; j++)
      if (s0 + j < steps) {
        b[j] = *reinterpret_cast<const u32x4_t*>(wat + 32 * (s0 + j));
        a[j] = *reinterpret_cast<const u32x4_t*>(xat + 32 * (s0 + j));
        if (!PACKED) a2[j] = *reinterpret_cast<const u32x4_t*>(xat + per_part + 32 * (s0 + j));
      }
#pragma unroll
    for (int j = 0; j < BATCH; j++)
      if (s0 + j < steps) {
        lower = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a[j]), __builtin_bit_cast(bf16x8_t, b[j]), lower, 0, 0, 0);
        if (!PACKED) upper = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a2[j]), __builtin_bit_cast(bf16x8_t, b[j]), upper, 0, 0, 0);
      }
  }
  // part[wave][register][lane]; lane (q, r16) of register i: activation row 4 q + i (PACKED: of part (4 q + i) / 8), column r16 & 7 of part r16 / 8
  const f32x4_t mine = PACKED || half == 0 ? lower : upper;
#pragma unroll
  for (int i = 0; i < 4; i++) part[(wave * 4 + i) * 64 + lane] = mine[i];
  __syncthreads();
  if (threadIdx.x < 16 * FRONT_COLUMNS) {
    const int row = threadIdx.x >> 3, c = threadIdx.x & 7, n = n0 + c;
    if (row < g.m && n < g.n) {
      float sum = 0.f;
      for (int w = 0; w < FRONT_WAVES; w++) {  // in the order of K
        const float* at = part + (w * 4 + (row & 3)) * 64;
        sum += at[16 * (row >> 2) + c];
        sum += at[16 * ((row >> 2) + (PACKED ? 2 : 0)) + 8 + c];
      }
      g.fused[(int64_t)row * g.n + n] = sum;
      if (n >= g.e) g.lat[(int64_t)row * (g.n - g.e) + n - g.e] = bf16_of(sum);
    }
  }
}
// The second launch: routing and plan of those rows - up to ROUTE_FUSED_ROWS of them by one workgroup, else a workgroup a row of which the
// last to arrive plans, as moe_plan_kernel and moe_route_plan_kernel do it - and beside them, in the workgroups past `groups`, the shared
// expert's up projection, which needs nothing of the routing: the plan leaves the memory and all but a few compute units idle.
// (18 and 9 registers a lane go to memory: the ranking's, as in moe_plan_kernel; the projection stays within the 128 of a workgroup of 1024.)
template <bool MANY>
__global__ __launch_bounds__(PLAN_THREADS) void latent_plan_kernel(RouteParams route, int rows, int by_rows, int e_lo, int e_n, int32_t* __restrict__ plan,
                                                                   int32_t* __restrict__ order, int slot_cap, int groups, StreamParams up) {
  extern __shared__ __align__(16) uint8_t rings[];
  int* lds = reinterpret_cast<int*>(rings);
  if ((int)blockIdx.x >= groups) {
    nvfp4_workgroup<EPI_DENSE_RELU2>(up, 0, blockIdx.x - groups, rings);
    return;
  }
  const int wave = threadIdx.x >> 6;
  bool cleared = false;
  if constexpr (MANY) {
    __shared__ int last;
    if (wave == 0) {
      route_any(route, blockIdx.x, threadIdx.x);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this row's ids (write-through stores) have reached memory before the ticket is drawn
    } else if (by_rows) {
      constexpr int IDLE = PLAN_THREADS - 64;
      clear_plan(plan, slot_cap, blockIdx.x * IDLE + (int)threadIdx.x - 64, groups * IDLE);
    }
    __syncthreads();
    if (threadIdx.x == 0) last = last_to_arrive(plan, groups);
    __syncthreads();
    if (!last) return;
    cleared = true;
  } else {
    if (wave < rows) route_any(route, wave, threadIdx.x & 63);
    __syncthreads();
  }
  if (by_rows) {
    plan_by_rows(route.ids, rows, route.k, e_lo, e_n, 0, plan, order, ROWS_PER_SLOT, slot_cap, lds, cleared);
  } else {
    plan_work<false>(route.ids, rows * route.k, e_lo, e_n, 0, plan, order, ROWS_PER_SLOT, slot_cap, nullptr, 1, 0, 0, lds);
  }
}

// experiments (hb_tune): the stream's workgroup shape ("nvfp4_ksplit", "nvfp4_nbw"); "nvfp4_tile": 1 forces the panel kernel, 2 the stream
static std::atomic<int> g_nvfp4_ksplit{0}, g_nvfp4_nbw{0}, g_nvfp4_tile{0}, g_nvfp4_few{0}, g_nvfp4_tile_ks{0}, g_nvfp4_lag{0}, g_nvfp4_fused{0};  // "nvfp4_fused": 1 runs fc1 and fc2 of a routed call on the stream in one launch, 2 (of any) in two; "nvfp4_lag": how far fc2 is behind in one, in units of eight slots; "nvfp4_few": 2 switches off the body for slots of at most eight rows; "nvfp4_tile_ks": the workgroups that share a tile's K

static int shape_nvfp4(StreamParams& p, int64_t busy_slots) {
  pick_shape(p.n_blocks, p.chunks, busy_slots, 4096, &p.ks, &p.nbw);
  if (g_nvfp4_ksplit) {
    p.ks = g_nvfp4_ksplit;
    p.nbw = g_nvfp4_nbw ? g_nvfp4_nbw.load() : 1;
  }
  if (p.ks * p.nbw > 16 || p.ks > p.chunks || (p.ks & (p.ks - 1))) return HB_EINVAL;
  set_split(p);
  p.no_few = g_nvfp4_few == 2;
  return HB_OK;
}

// The shape of a dense call of one slot: K split eight ways as far as there are chunks, since a wavefront's start and the
// exchange cost about as much as two or three of them. Measured, replayed graphs of calls on cycled weights, the general rule and
// this one (us, blocks x chunks): twelve rows 16 x 12 10.8 and 5.4, 160 x 12 12.0 and 6.0, 400 x 16 12.5 and 10.9, 640 x 4 8.3 and
// 6.8, 800 x 8 13.2 and 10.9; eight rows 80 x 12 8.2 and 5.6, 400 x 16 10.4 and 9.5, 640 x 12 13.2 and 10.8; one row 80 x 4 4.9 and
// 4.4. With few rows and many blocks short of K the launch is bound by its traffic, and fewer wavefronts are better:
// - 257 to 512 blocks, where the general rule's workgroups of two blocks all start at once: its shape up to two rows below sixteen
//   chunks (the splits took 0.95 to 1.11 times as long: 302 x 10 1.11, 400 x 8 1.07, 300 x 12 1.06) and, past 300 blocks, up to
//   eight rows below twelve (0.96 to 1.06);
// - 513 to 767 blocks: its shape below eight chunks (640 x 7 one row 7.0, split four ways 7.8), four ways below twelve (520 x 8
//   one row by the general rule 8.4, split eight ways 9.0, four ways 8.2);
// - from three blocks a compute unit its shape: four blocks a workgroup took 1.21 times as long at 768 x 40 and eight rows, 1200 x
//   40 1.38, 2374 x 24 1.12, and gained at 800 blocks alone (one row up to 11 %).
static void shape_nvfp4_dense(StreamParams& p) {
  constexpr int COMPUTE_UNITS = 256;
  int most = 8;
  if (p.m <= FP4_FEW_ROWS && !p.no_few && p.n_blocks > COMPUTE_UNITS) {
    if (p.n_blocks <= 2 * COMPUTE_UNITS) {
      if (p.chunks < (p.m <= 2 ? 16 : p.n_blocks > 300 ? 12 : 0)) return;
    } else if (p.n_blocks < 3 * COMPUTE_UNITS && p.chunks >= 8) {
      most = p.chunks < 12 ? 4 : 8;
    } else {
      return;
    }
  }
  while (p.ks < most && 2 * p.ks <= p.chunks) p.ks *= 2;
  if (p.ks >= 4) p.nbw = 1;
  set_split(p);
}

// Blocks, times slots of sixteen rows, up to which a dense call gives a block's tiles to two workgroups (up to half of them: to four).
constexpr int FP4_PARTS_BLOCKS = 128;
template <int EPI>
static int launch_nvfp4(StreamParams& p, int64_t slots, int64_t busy_slots, hipStream_t stream) {
  if (int e = shape_nvfp4(p, busy_slots)) return e;
  if (epi_dense(EPI) && slots == 1 && !g_nvfp4_ksplit) shape_nvfp4_dense(p);
  if constexpr (epi_dense(EPI)) {
    if (!g_nvfp4_ksplit && p.n_blocks * slots <= FP4_PARTS_BLOCKS) {
      p.nbw = 1;
      const int most = p.m > FP4_FEW_ROWS && p.chunks >= 24 ? 16 : 8;  // a wavefront's start and the exchange against the expansion of nine rows and more
      while (p.ks < most && 2 * p.ks <= p.chunks) p.ks *= 2;
      set_split(p);
      const bool four = p.n_blocks * slots <= FP4_PARTS_BLOCKS / 2;
      const dim3 grid((unsigned)((p.n_blocks + 7) / 8 * 8 * (four ? 4 : 2)), (unsigned)slots);
      auto launch = [&](auto kernel) { HB_LAUNCH(kernel, grid, dim3(64 * p.ks), (size_t)p.ks * FP4_RING_BYTES, stream, p); };
      four ? launch(nvfp4_part_kernel<EPI, 4>) : launch(nvfp4_part_kernel<EPI, 2>);
      return HB_OK;
    }
  }
  const dim3 grid((unsigned)((p.n_blocks + p.nbw - 1) / p.nbw), (unsigned)slots);
  const int waves = p.ks * p.nbw;
  HB_LAUNCH(nvfp4_stream_kernel<EPI>, grid, dim3(64 * waves), (size_t)waves * FP4_RING_BYTES, stream, p);
  return HB_OK;
}

// The shape of the dense `b` beside the shaped `a` in one launch: one workgroup size (and LDS a workgroup) for both, which the plan's matrix sets. A small
// latent block's shared expert has these splits of K in every form, so that its bits do not depend on the form.
static int shape_beside(StreamParams& b, int64_t slots_b, const StreamParams& a) {
  if (int e = shape_nvfp4(b, slots_b)) return e;
  const int waves = a.ks * a.nbw;
  b.ks = std::min(b.ks, waves);
  b.nbw = waves / b.ks;
  set_split(b);
  return HB_OK;
}

// `a` over its plan's slots beside the dense `b` in one launch (nvfp4_twin_kernel).
template <int EPI_A, int EPI_B>
static int launch_twin(StreamParams& a, int64_t slots_a, int64_t busy_a, StreamParams& b, int64_t slots_b, hipStream_t stream) {
  if (int e = shape_nvfp4(a, busy_a)) return e;
  if (int e = shape_beside(b, slots_b, a)) return e;
  const int groups_a = (a.n_blocks + a.nbw - 1) / a.nbw, groups_b = (b.n_blocks + b.nbw - 1) / b.nbw;
  const int64_t first = slots_b * groups_b, all = first + slots_a * groups_a;
  if (all > 0x7fffffff) return HB_EINVAL;
  const int waves = std::max(a.ks * a.nbw, b.ks * b.nbw);
  HB_LAUNCH((nvfp4_twin_kernel<EPI_A, EPI_B>), dim3((unsigned)all), dim3(64 * waves), (size_t)waves * FP4_RING_BYTES, stream, a, b, groups_a, groups_b, (int)first);
  return HB_OK;
}

// Whether the two layers share a launch. The one launch fills the compute units that a round of fc1's workgroups leaves idle when it
// ends, and pays for it with a trip of h's arrival counters through memory, about a microsecond longer than the boundary between
// two launches. So it needs about as many wavefronts as the device holds (4096), or a quarter of that where a wavefront has four chunks and more, and it
// loses again over many rounds of slots of unequal length (the order of the grid then holds fc2 back). Measured, the two launches and the one, replayed
// graphs of calls with changing routing, us, experts (latent, inter) and pairs:
// - too few: 128 (512, 1024) 32 20.8 and 23.5, 320 31.4 and 34.9; 256 (768, 1536) 48 23.2 and 24.3; 160 (512, 1536) 192 35.1 and 37.5;
// - 256 (768, 1536) 192 49.4 and 46.5; 512 (768, 1024) 256 51.4 and 47.1, 640 75.4 and 71.4; 512 (512, 2688) 176 61.7 and 58.2;
// - eight chunks of K and more: 384 (1024, 2048) 16 38.5 and 37.8 (whole block), 64 48.0 and 43.5, 256 91.4 and 85.7; 512 (1024, 2688) 22 32.3 and 32.0, 88
//   63.4 and 58.1, 352 152.4 and 147.7; 128 (1024, 1024) 320 43.3 and 38.9;
// - too many: 384 (1024, 2048) 384 113.2 and 116.4; 512 (512, 2688) 880 131.3 and 136.5; 256 (768, 1536) 1440 86.8 and 90.6;
// - more than two rows an expert, even and (skewed) routing: 128 (1024, 2048) 384 65.3 and 66.1 (60.7 and 64.4), 640 75.6 and 77.1 (70.8 and 74.8), but 128 (1024, 1024) 384
//   42.7 and 38.2 (40.1 and 35.9), 64 (2048, 2048) 252 67.6 and 64.4 (66.4 and 66.8);
// - a row an expert and K of fc1 below six chunks: 160 (512, 1536) 320 41.4 and 41.2 (38.7 and 42.4); 300 (640, 1280) 300 46.6 and 46.1 (42.4 and 44.6), 900 66.6 and
//   66.4 (57.1 and 58.3); fewer pairs of few blocks: 512 (512, 1024) 256 40.0 and 38.9 (34.8 and 39.4), of many 512 (512, 2688) 176 61.1 and 57.5 (50.1 and 48.3);
// - of six and seven chunks even routing, as this path's is, gains and skewed routing loses: 256 (768, 1536) 252 52.8 and 51.2 (47.4 and 50.1), 512 (768, 1024) 250 48.2
//   and 43.7 (40.4 and 44.5);
// - K of fc2 past 24 chunks, whose few long workgroups meet on one compute unit: 8 (2048, 5632) 16 28.5 and 34.2 (28.4 and 32.0), 32 31.6 and 37.1; 16 (1024, 8192) 8 25.8 and 28.3 (25.9 and
//   29.0); 32 (2048, 4096) 64 60.9 and 57.5 (57.5 and 61.4), 96 62.7 and 58.5 (59.7 and 64.3).
constexpr int DEVICE_WAVES = 4096;
// `local`: the experts held here, of the `experts` that the pairs name; p1, p2: the layers.
static bool fc12_serves(int64_t pairs, int local, int64_t experts, const StreamParams& p1, const StreamParams& p2) {
  if (g_nvfp4_fused) return g_nvfp4_fused == 1;
  if (p2.chunks > 24) return false;
  const bool deep = p1.chunks >= 8;
  const double distinct = local * (1.0 - std::exp(-(double)pairs / (double)experts));  // of a uniform routing
  const double waves = distinct * p1.n_blocks * (deep ? 2 : 1);
  if (waves < (deep ? DEVICE_WAVES / 4 : p1.chunks >= 6 ? DEVICE_WAVES * 3 / 4 : DEVICE_WAVES)) return false;
  return pairs < experts || (waves <= 2 * DEVICE_WAVES && pairs <= 2 * experts && p1.chunks >= 6) || (deep && waves <= DEVICE_WAVES);
}

// Both layers over a plan of `slots` entries (busy: the caller's estimate of those with rows), in one launch; `dense`: one slot of a dense matrix
// beside them, or null.
template <int EPI1>
static int launch_fc12(StreamParams& p1, StreamParams& p2, int64_t slots, int64_t busy, StreamParams* dense, hipStream_t stream) {
  if (!fc12_apart(p1)) return HB_EINVAL;  // (the caller then takes two)
  if (int e = shape_nvfp4(p1, busy)) return e;
  if (int e = shape_nvfp4(p2, busy)) return e;
  const int waves = std::max(p1.ks * p1.nbw, p2.ks * p2.nbw);  // one workgroup size for both: all powers of two
  int first = 0;
  if (dense) {
    if (int e = shape_beside(*dense, 1, p2)) return e;
    dense->nbw = waves / dense->ks;
    first = (dense->n_blocks + dense->nbw - 1) / dense->nbw;
  }
  p1.nbw = waves / p1.ks;
  p2.nbw = waves / p2.ks;
  const int groups1 = (p1.n_blocks + p1.nbw - 1) / p1.nbw, groups2 = (p2.n_blocks + p2.nbw - 1) / p2.nbw;
  const int64_t total = slots * (groups1 + groups2) + first;
  if (total > 0x7fffffff) return HB_EINVAL;
  moe_await_slots(p1, p2, const_cast<int32_t*>(p1.plan), slots, groups1);
  // about half the device's workgroups ahead (1024 (4 wavefronts) started at once, twice that: 512 (1024, 2688) at 176 pairs 32 slots 91.7 us, 48 89.2, 96 88.4)
  const int lag = (int)std::min<int64_t>(slots, g_nvfp4_lag ? 8 * g_nvfp4_lag.load() : std::max(8, 2048 / groups1));
  HB_LAUNCH(nvfp4_fc12_kernel<EPI1>, dim3((unsigned)total), dim3(64 * waves), (size_t)waves * FP4_RING_BYTES, stream, p1, p2, dense ? *dense : StreamParams{}, groups1,
            groups2, (int)slots, lag, first);
  return HB_OK;
}

static int launch_front(const LatentRouter& r, hipStream_t stream) {
  const int n = r.experts + r.latent;
  if (r.m <= 0 || r.m > LATENT_MAX_ROWS || r.hidden <= 0 || r.hidden % 512 || r.latent < 0 || r.steps <= 0) return HB_EINVAL;
  const FrontGemv g{r.w, r.x, r.fused, r.lat, n, r.hidden, r.m, r.experts};
  const dim3 grid((unsigned)((n + FRONT_COLUMNS - 1) / FRONT_COLUMNS));
  auto launch = [&](auto kernel) { HB_LAUNCH(kernel, grid, dim3(64 * FRONT_WAVES), 0, stream, g); };
  r.m <= 8 ? launch(latent_front_kernel<true>) : launch(latent_front_kernel<false>);
  return HB_OK;
}

// Routing and plan beside `up` (latent_plan_kernel), whose splits of K are those of the launch beside `fc1`.
static int launch_latent_plan(const LatentRouter& r, const LatentPlan& q, StreamParams& up, const StreamParams& fc1, hipStream_t stream) {
  if (int e = shape_beside(up, 1, fc1)) return e;
  up.nbw = 1;
  const size_t lds = std::max(q.lds, (size_t)up.ks * FP4_RING_BYTES);
  auto launch = [&](auto kernel) {
    HB_LAUNCH(kernel, dim3((unsigned)(q.groups + up.n_blocks)), dim3(PLAN_THREADS), lds, stream, q.route, r.m, q.by_rows, r.e_lo, r.e_n, r.ws->plan, r.ws->order, q.slot_cap,
              q.groups, up);
  };
  q.groups > 1 ? launch(latent_plan_kernel<true>) : launch(latent_plan_kernel<false>);
  return HB_OK;
}

// ------------------------------------------------------------------------------ the panel kernel's NVFP4 format
struct TileNvfp4 {
  typedef Fp4Chunk Chunk;
  typedef Fp4Ring Ring;
  struct Part {  // a fragment being expanded: its eight codes and their block's scale
    uint32_t codes;
    float scale;
  };
  template <int NT, int S>
  static __device__ __forceinline__ Part open(const Chunk& ch, const Slot&) {
    return Part{ch.tile(NT)[S], fp4_scale<S>(ch.sc[NT])};
  }
#define HB_FP4_CVT "v_cvt_scalef32_pk_f32_fp4"
  template <int K, bool AFTER_VALU>  // a product, then values 2 K, 2 K + 1 of the part
  static __device__ __forceinline__ void product_pair(f32x4_t& acc, const u32x4_t& w, const u32x4_t& a, const Part& part, uint32_t& out) {
    if constexpr (K == 0 && AFTER_VALU) HB_PANEL_PRODUCT_PAIR("s_nop 1\n\t", HB_FP4_CVT, "", acc, out, w, part.codes, part.scale, a);
    if constexpr (K == 0 && !AFTER_VALU) HB_PANEL_PRODUCT_PAIR("", HB_FP4_CVT, "", acc, out, w, part.codes, part.scale, a);
    if constexpr (K == 1) HB_PANEL_PRODUCT_PAIR("", HB_FP4_CVT, " op_sel:[1,0,0]", acc, out, w, part.codes, part.scale, a);
    if constexpr (K == 2) HB_PANEL_PRODUCT_PAIR("", HB_FP4_CVT, " op_sel:[0,1,0]", acc, out, w, part.codes, part.scale, a);
    if constexpr (K == 3) HB_PANEL_PRODUCT_PAIR("", HB_FP4_CVT, " op_sel:[1,1,0]", acc, out, w, part.codes, part.scale, a);
  }
  template <int K, bool AFTER_VALU>  // a product, then the first half of that
  static __device__ __forceinline__ void product_first(f32x4_t& acc, const u32x4_t& w, const u32x4_t& a, const Part& part, panel_two_t& two) {
    if constexpr (K == 0 && AFTER_VALU) HB_PANEL_PRODUCT_FIRST("s_nop 1\n\t", HB_FP4_CVT, "", acc, two, w, part.codes, part.scale, a);
    if constexpr (K == 0 && !AFTER_VALU) HB_PANEL_PRODUCT_FIRST("", HB_FP4_CVT, "", acc, two, w, part.codes, part.scale, a);
    if constexpr (K == 1) HB_PANEL_PRODUCT_FIRST("", HB_FP4_CVT, " op_sel:[1,0,0]", acc, two, w, part.codes, part.scale, a);
    if constexpr (K == 2) HB_PANEL_PRODUCT_FIRST("", HB_FP4_CVT, " op_sel:[0,1,0]", acc, two, w, part.codes, part.scale, a);
    if constexpr (K == 3) HB_PANEL_PRODUCT_FIRST("", HB_FP4_CVT, " op_sel:[1,1,0]", acc, two, w, part.codes, part.scale, a);
  }
  template <int K>
  static __device__ __forceinline__ void pair_alone(const Part& part, uint32_t& out) {
    if constexpr (K == 0) HB_PANEL_PAIR_ALONE(HB_FP4_CVT, "", out, part.codes, part.scale);
    if constexpr (K == 1) HB_PANEL_PAIR_ALONE(HB_FP4_CVT, " op_sel:[1,0,0]", out, part.codes, part.scale);
    if constexpr (K == 2) HB_PANEL_PAIR_ALONE(HB_FP4_CVT, " op_sel:[0,1,0]", out, part.codes, part.scale);
    if constexpr (K == 3) HB_PANEL_PAIR_ALONE(HB_FP4_CVT, " op_sel:[1,1,0]", out, part.codes, part.scale);
  }
  static constexpr int BLOCK_BYTES = NVFP4_BLOCK_BYTES;
  static constexpr bool PER_ROW = false;
  static constexpr float EXPAND_US = 0.f;  // (the estimate's own constants are this format's)
  static constexpr int BESIDE_TILES = 0;
  static constexpr int LOW_ROWS = 24, MIDDLE_ROWS = 46, MIDDLE_ROWS_LARGE = 46, HIGH_ROWS = 70;  // panel_height's lines
  static constexpr int LIGHT_ROWS = 0;  // (an expansion takes the scale along at the price of the stream's)
  template <int EPI, class Wait>
  static __device__ __forceinline__ void light(const StreamParams&, const Slot&, int, uint8_t*, Wait&) {}
};

static inline unsigned grid_for(int64_t threads) { return (unsigned)((threads + 255) / 256); }

}  // namespace hb

using namespace hb;

static StreamParams dense_params(const void* tiled, float scale, int n, int k, const void* x, int m, void* y) {
  StreamParams p{};
  p.w = static_cast<const uint8_t*>(tiled);
  p.scalar = scale;
  p.n_blocks = n / 64;
  p.chunks = k / 128;
  p.a = static_cast<const uint16_t*>(x);
  p.a_stride = k;
  p.m = m;
  p.out = y;
  p.out_stride = n;
  return p;
}

extern "C" size_t hb_nvfp4_tiled_bytes(int64_t rows, int k) {
  if (rows <= 0 || k <= 0 || rows % 64 || k % 128) return 0;
  return (size_t)(rows / 64) * (size_t)(k / 128) * NVFP4_BLOCK_BYTES;
}

extern "C" int hb_nvfp4_repack(const uint8_t* weight, const uint8_t* scales, int swizzled, int64_t rows, int k, void* tiled, void* stream) {
  if (!weight || !scales || !tiled) return HB_ENULL;
  if (rows <= 0 || k <= 0 || rows % 64 || k % 128) return HB_EINVAL;
  const int chunks = k / 128;
  const int64_t blocks = rows / 64 * chunks;
  hipLaunchKernelGGL(nvfp4_repack_codes_kernel, dim3(grid_for(blocks * 256)), dim3(256), 0, as_stream(stream), weight, blocks, chunks,
                     static_cast<uint8_t*>(tiled));
  hipLaunchKernelGGL(nvfp4_repack_scales_kernel, dim3(grid_for(blocks * 512)), dim3(256), 0, as_stream(stream), scales, swizzled, blocks, chunks,
                     static_cast<uint8_t*>(tiled));
  return launch_status();
}

extern "C" int hb_nvfp4_dequant(const void* tiled, float global_scale, int64_t rows, int k, float* out, void* stream) {
  if (!tiled || !out) return HB_ENULL;
  if (rows <= 0 || k <= 0 || rows % 64 || k % 128) return HB_EINVAL;
  const int chunks = k / 128;
  const int64_t blocks = rows / 64 * chunks;
  hipLaunchKernelGGL(nvfp4_dequant_kernel, dim3(grid_for(blocks * 256)), dim3(256), 0, as_stream(stream), static_cast<const uint8_t*>(tiled),
                     global_scale, blocks, chunks, out);
  return launch_status();
}

// The weight stream passes over the matrix once for every sixteen rows; the panel kernel expands it once for 128, and is the
// faster one past sixteen rows except on few blocks. Measured, stream and panel, replayed graphs, us:
// - Up to FP4_PARTS_BLOCKS blocks times passes, whose workgroups share each block's tiles (nvfp4_part_kernel), the stream is the faster
//   one: 64 blocks x 8 chunks 32 rows 4.5 and 6.2, x 16 17 rows 5.8 and 8.7, x 40 10.0 and 16.0; 16 blocks x 24 128 rows 6.9 and 10.9; 8 blocks x
//   64 256 rows 13.7 and 18.6. Past 64 chunks the panel's cut with K shared among workgroups takes over (8 blocks x 100 17 rows 15.8 and
//   13.2, 64 blocks x 160 17 rows 33.1 and 26.1). Fewer than eight blocks leave compute dies idle, whose L2s would serve the rows of many passes: one
//   block x 24 128 rows 6.2 and 10.6, 500 rows 18.4 and 10.8; x 48 128 rows 9.2 and 9.7, x 64 11.1 and 10.8.
// - Up to 256, whole blocks a workgroup, where K is long and the cut shares no tile's K: the stream splits K sixteen ways in a workgroup
//   where the panel has eight. 32 blocks x 32 chunks 128 rows 11.2 and 13.6, x 28 12.6 and 12.3, x 16 8.7 and 8.6, x 8 8.8 and 6.1; 80 blocks x 40
//   48 rows (240 workgroups) 13.8 and 15.7, 64 rows (320) 22.3 and 13.6.
constexpr int STREAM_LONG_CHUNKS = 32, STREAM_PASSES_WORKGROUPS = 256, DIES = 8;
static bool stream_serves(int m, int n_blocks, int chunks, const PanelPlan& cut) {
  const int64_t passes = (m + ROWS_PER_SLOT - 1) / ROWS_PER_SLOT;
  if (n_blocks * passes <= FP4_PARTS_BLOCKS && (n_blocks >= DIES ? chunks <= 64 : chunks <= 48 && passes <= 8)) return true;
  return cut.kz == 1 && chunks >= STREAM_LONG_CHUNKS && n_blocks * passes <= STREAM_PASSES_WORKGROUPS;
}
static PanelForce nvfp4_force() { return PanelForce{g_nvfp4_ksplit, g_nvfp4_nbw, g_nvfp4_tile_ks}; }

// `workspace`: room for partial tiles (hb_nvfp4_gemm_room_bytes), or null: no call shares K among workgroups.
static int nvfp4_gemm(const void* x, int m, const void* tiled, float global_scale, int n, int k, int relu2, void* y, void* workspace, size_t workspace_bytes,
                      hipStream_t stream) {
  if (!x || !tiled || !y) return HB_ENULL;
  if (m <= 0 || n <= 0 || k <= 0 || n % 64 || k % 128) return HB_EINVAL;
  if (!aligned(x, 16) || !aligned(tiled, 16) || !aligned(y, 2) || !aligned(workspace, 16)) return HB_EINVAL;
  StreamParams p = dense_params(tiled, global_scale, n, k, x, m, y);
  if (panel_takes(m, k) && panel_writes(y, false) && (g_nvfp4_tile == 1 || (g_nvfp4_tile == 0 && m > ROWS_PER_SLOT))) {
    const PanelForce force = nvfp4_force();
    const PanelPlan cut = cut_panel<TileNvfp4>(m, p.n_blocks, p.chunks, workspace ? workspace_bytes : 0, force);
    if (g_nvfp4_tile == 1 || force.ks || force.kz || !stream_serves(m, p.n_blocks, p.chunks, cut)) {
      if (int e = relu2 ? launch_panel<TileNvfp4, EPI_DENSE_RELU2>(p, cut, workspace, stream) : launch_panel<TileNvfp4, EPI_DENSE>(p, cut, workspace, stream)) return e;
      return launch_status();
    }
  }
  const int64_t slots = (m + ROWS_PER_SLOT - 1) / ROWS_PER_SLOT;
  if (slots > 65535) return HB_EINVAL;
  if (int e = relu2 ? launch_nvfp4<EPI_DENSE_RELU2>(p, slots, slots, stream) : launch_nvfp4<EPI_DENSE>(p, slots, slots, stream)) return e;
  return launch_status();
}

extern "C" int hb_nvfp4_gemm(const void* x, int m, const void* tiled, float global_scale, int n, int k, int relu2, void* y, void* stream) {
  return nvfp4_gemm(x, m, tiled, global_scale, n, k, relu2, y, nullptr, 0, as_stream(stream));
}

// Kept for callers built against it: room for every tile of four blocks (128 rows) to have its K shared by about four hundred
// workgroups in all, which no cut needs any more; a call takes the best cut that fits what it is given. New callers ask
// hb_nvfp4_gemm_room_bytes, which is what the best cut uses.
extern "C" size_t hb_nvfp4_gemm_workspace_bytes(int m, int n, int k) {
  if (m <= 20 || n <= 0 || k <= 0 || n % 64 || k % 128) return 0;
  const int64_t tiles = (int64_t)((n / 64 + 3) / 4) * ((m + 127) / 128), chunks = k / 128;
  const int64_t ks = g_nvfp4_tile_ks ? std::min<int64_t>(g_nvfp4_tile_ks, chunks) : tiles >= 200 ? 1 : std::max<int64_t>(1, std::min<int64_t>(chunks / 4, 400 / tiles));
  const int mt = (std::min(m, 128) + 15) / 16;
  return ks > 1 ? (((size_t)(PLAN_HEADER + tiles) * sizeof(uint32_t) + 255) & ~(size_t)255) + (size_t)tiles * ks * 4 * mt * 4 * 64 * sizeof(f32x4_t) : 0;
}

extern "C" size_t hb_nvfp4_gemm_room_bytes(int m, int n, int k) {
  if (m <= ROWS_PER_SLOT || n <= 0 || k <= 0 || n % 64 || k % 128) return 0;
  const PanelForce force = nvfp4_force();
  const PanelPlan cut = cut_panel<TileNvfp4>(m, n / 64, k / 128, PANEL_ANY_ROOM, force);
  return g_nvfp4_tile == 0 && !force.ks && !force.kz && stream_serves(m, n / 64, k / 128, cut) ? 0 : panel_room(cut);
}

extern "C" int hb_nvfp4_gemm_ws(const void* x, int m, const void* tiled, float global_scale, int n, int k, int relu2, void* y, void* workspace,
                                size_t workspace_bytes, void* stream) {
  return nvfp4_gemm(x, m, tiled, global_scale, n, k, relu2, y, workspace_bytes ? workspace : nullptr, workspace_bytes, as_stream(stream));
}

// ------------------------------------------------------------------------------------------------ routed experts
namespace {


int check_experts(const hb_nvfp4_experts* ex) {
  if (!ex) return HB_ENULL;
  if (!ex->fc1 || !ex->fc1_scale2 || !ex->fc2 || !ex->fc2_scale2) return HB_ENULL;
  if (ex->experts <= 0 || ex->hidden <= 0 || ex->inter <= 0 || ex->hidden_out <= 0) return HB_EINVAL;
  const int n1 = ex->gated ? 2 * ex->inter : ex->inter;
  if (ex->hidden % 128 || ex->inter % 128 || n1 % 64 || ex->hidden_out % 64) return HB_EINVAL;
  if (!aligned(ex->fc1, 16) || !aligned(ex->fc2, 16) || !aligned(ex->fc1_scale2, 4) || !aligned(ex->fc2_scale2, 4)) return HB_EINVAL;
  return HB_OK;
}

// The two launches' parameters of a routed call over a filled plan: fc1 from x into ws.h, fc2 from there into `out_pairs`.
void expert_params(const hb_nvfp4_experts* ex, const void* x, int m, int topk, const MoeWorkspace& ws, void* out_pairs, int pairs_bf16, StreamParams& p,
                   StreamParams& f2) {
  const int64_t pairs = (int64_t)m * topk;
  const int n1 = ex->gated ? 2 * ex->inter : ex->inter;
  p = StreamParams{};
  p.w = static_cast<const uint8_t*>(ex->fc1);
  p.expert_bytes = (int64_t)hb_nvfp4_tiled_bytes(n1, ex->hidden);
  p.scalars = ex->fc1_scale2;
  p.n_blocks = n1 / 64;
  p.chunks = ex->hidden / 128;
  p.a = static_cast<const uint16_t*>(x);
  p.a_stride = ex->hidden;
  p.plan = ws.plan;
  p.order = ws.order;
  p.topk = topk;
  p.pairs = (int)pairs;
  p.out = ws.h;
  p.out_stride = ex->inter;
  f2 = p;
  f2.w = static_cast<const uint8_t*>(ex->fc2);
  f2.expert_bytes = (int64_t)hb_nvfp4_tiled_bytes(ex->hidden_out, ex->inter);
  f2.scalars = ex->fc2_scale2;
  f2.n_blocks = ex->hidden_out / 64;
  f2.chunks = ex->inter / 128;
  f2.a = ws.h;
  f2.a_stride = ex->inter;
  f2.out = out_pairs;
  f2.out_stride = ex->hidden_out;
  f2.out_bf16 = pairs_bf16;
}

// the slots the stream's shape is chosen for: a call of few pairs fills about one slot a distinct expert
int64_t busy_slots(int64_t pairs, int experts, int64_t slots) { return pairs < 2 * experts ? (pairs + 1) / 2 : slots; }

// plan -> fc1 -> fc2: `out_pairs` receives fc2's per-pair outputs.
int run_experts(const hb_nvfp4_experts* ex, const void* x, const int32_t* ids, int m, int topk, const MoeWorkspace& ws, void* out_pairs,
                int pairs_bf16, hipStream_t stream, int experts_total) {
  const int64_t pairs = (int64_t)m * topk, named = experts_named(experts_total, ex->base, ex->experts);
  // A dense contraction once an expert sees three rows, or four of fewer than 768 columns: the panel kernel; below that the 16-row slots of the weight
  // stream. Measured, stream and panel, the whole latent block in us: 300 (640, 1280) 3 rows an expert 89 and 90, 4 rows 94 and 90; 256 (768, 1536) 3 rows 97 and 96, 5 rows
  // 106 and 102; 400 (896, 2048) 3 rows 180 and 175, 5 rows 202 and 190; 512 (1024, 2688) 3 rows 294 and 286, 5 rows 338 and 318, 7 rows 373 and 339.
  // Few experts fill the device later: with fc1 (`fill`: its workgroups, a slot an expert), and with fc2, whose workgroups (`fill2`) are as long as their K. By fill2 a chunk of K,
  // the routed call, even and (skewed) routing, us:
  // - 32 to 50: 64 (2048, 2048) 4 rows 63 and 67 (66 and 68), 5 rows 71 and 68 (71 and 69); 128 (1024, 2048) 3 rows 65 and 73 (65 and 64), 5 rows 78 and 74 (76 and 73); 200 (896,
  //   2048) 4 rows 93 and 93 (83 and 85), 6 rows 99 and 96 (98 and 93);
  // - 12 to 26: 160 (512, 1536) 5 rows 48 and 51 (47 and 47), 7 rows 52 and 52 (52 and 54); 96 (1024, 4096) 5 rows 97 and 107 (90 and 108), 8 rows 114 and 110 (118 and 115);
  // - 4 to 9: 48 (768, 2816) 8 rows 50 and 53 (51 and 55), 12 rows 56 and 54 (58 and 56); 32 (1024, 2688) 12 rows 47 and 51 (49 and 55), 20 rows 56 and 53 (56 and 58); 64 (1024, 8192) 10
  //   rows 150 and 153 (159 and 175), 16 rows 203 and 155 (206 and 192);
  // - 1: 16 (1024, 8192) 4 rows 42 and 100 (45 and 100), 40 rows 110 and 125 (109 and 131), 64 rows 159 and 136 (155 and 164).
  // Too few workgroups for a round of both layers leave it to the stream: 8 (2048, 2048) 12 rows 28 and 51, 120 rows 78 and 87, 150 rows
  // 103 and 88; 16 (512, 1024) 40 rows 27 and 32, 120 rows 39 and 44.
  // A range of the experts sees its share of the pairs only: 64 of 512 experts (1024, 2688), the summed experts alone, two launches, on slots of 128 rows 4
  // rows an expert 59 and 68, 8 rows 86 and 76.
  const int64_t fill = (int64_t)ex->experts * (((ex->gated ? 2 : 1) * ex->inter / 64 + 3) / 4), fill2 = (int64_t)ex->experts * ((ex->hidden_out / 64 + 3) / 4), chunks2 = ex->inter / 128;
  int64_t rows_min = fill2 >= 60 * chunks2 ? ex->hidden >= 768 ? 3 : 4 : fill2 >= 30 * chunks2 ? 5 : fill2 >= 10 * chunks2 ? 7 : fill2 >= 3 * chunks2 ? 14 : 60;
  if (fill < 500) rows_min = std::max<int64_t>(rows_min, 7);
  if (fill + fill2 < 256) rows_min = std::max<int64_t>(rows_min, 128);
  if (ex->experts < named) rows_min = 8;
  const bool dense = panel_takes(m, ex->hidden) && panel_takes(pairs, ex->inter) && panel_writes(out_pairs, !pairs_bf16) &&
                     (g_nvfp4_tile == 1 || (g_nvfp4_tile == 0 && pairs >= rows_min * named));
  const int tiles = panel_height<TileNvfp4>(pairs, named, ex->experts, 0, (ex->gated ? 2 : 1) * ex->inter / 64), slot_rows = dense ? 16 * tiles : ROWS_PER_SLOT;
  const int64_t slots = moe_max_slots(pairs, ex->experts, 0, slot_rows);
  if (moe_max_slots(pairs, ex->experts, 0, std::min(slot_rows, PANEL_REFUSED_ROWS)) > PANEL_MAX_SLOTS) return HB_EINVAL;
  if (int e = moe_launch_plan(ids, pairs, ex->base, ex->experts, 0, ws, stream, slot_rows)) return e;
  const int64_t est = busy_slots(pairs, ex->experts, slots);
  StreamParams p, f2;
  expert_params(ex, x, m, topk, ws, out_pairs, pairs_bf16, p, f2);
  if (dense && g_nvfp4_fused != 2 && fc12_apart(p) && (g_nvfp4_fused == 1 || panel_together(p, f2, ex->experts, tiles))) {
    if (int e = ex->gated ? launch_panel_fc12<TileNvfp4, EPI_FC1_GATED>(p, f2, ws.plan, tiles, slots, m, pairs, g_nvfp4_lag, stream)
                          : launch_panel_fc12<TileNvfp4, EPI_FC1_RELU2>(p, f2, ws.plan, tiles, slots, m, pairs, g_nvfp4_lag, stream))
      return e;
    return launch_status();
  }
  if (dense) {
    if (int e = ex->gated ? launch_panel_routed<TileNvfp4, EPI_FC1_GATED>(p, tiles, slots, m, stream) : launch_panel_routed<TileNvfp4, EPI_FC1_RELU2>(p, tiles, slots, m, stream)) return e;
    if (int e = launch_panel_routed<TileNvfp4, EPI_FC2>(f2, tiles, slots, pairs, stream)) return e;
    return launch_status();
  }
  if (fc12_serves(pairs, ex->experts, named, p, f2) && (ex->gated ? launch_fc12<EPI_FC1_GATED>(p, f2, slots, est, nullptr, stream) : launch_fc12<EPI_FC1_RELU2>(p, f2, slots, est, nullptr, stream)) == HB_OK)
    return launch_status();
  if (int e = ex->gated ? launch_nvfp4<EPI_FC1_GATED>(p, slots, est, stream) : launch_nvfp4<EPI_FC1_RELU2>(p, slots, est, stream)) return e;
  if (int e = launch_nvfp4<EPI_FC2>(f2, slots, est, stream)) return e;
  return launch_status();
}

// ------------------------------------------------------------------------------------- the small latent block
struct LatentWorkspace {
  MoeWorkspace moe;    // the routed experts' (absent without NVFP4 experts)
  uint16_t* routed;    // BF16 [m, latent]: the routed sum
  uint16_t* shared_h;  // BF16 [m, shared_inter]
  uint16_t* shared_y;  // BF16 [m, hidden]
  size_t bytes;
};

LatentWorkspace latent_carve(const hb_latent_weights* w, void* base, int m, int topk) {
  LatentWorkspace l{};
  size_t off = 0;
  if (w->routed) {
    l.moe = moe_carve(base, m, topk, w->routed->experts, w->routed->inter, w->routed->hidden_out, 0);
    off = l.moe.bytes;
  }
  auto take = [&](size_t bytes) {
    void* ptr = base ? static_cast<char*>(base) + off : nullptr;
    off += (bytes + 255) & ~(size_t)255;
    return static_cast<uint16_t*>(ptr);
  };
  l.routed = take((size_t)m * w->latent * 2);
  l.shared_h = take((size_t)m * w->shared_inter * 2);
  l.shared_y = take((size_t)m * w->hidden * 2);
  l.bytes = off;
  return l;
}

int check_latent(const hb_latent_weights* w, int m, int topk) {
  if (!w) return HB_ENULL;
  if (!w->gate_fc1 || !w->bias || !w->fc2) return HB_ENULL;
  if (m <= 0 || m > LATENT_MAX_ROWS || topk <= 0) return HB_EINVAL;
  if (w->experts_total <= 0 || w->latent <= 0 || w->hidden <= 0 || w->latent % 128 || w->hidden % 512) return HB_EINVAL;
  if (!aligned(w->gate_fc1, 16) || !aligned(w->fc2, 16) || !aligned(w->bias, 4)) return HB_EINVAL;
  if (w->routed) {
    if (int e = check_experts(w->routed)) return e;
    if (w->routed->hidden != w->latent || w->routed->hidden_out != w->latent || w->routed->base + w->routed->experts > w->experts_total) return HB_EINVAL;
  }
  if ((w->shared_up != nullptr) != (w->shared_down != nullptr)) return HB_ENULL;
  if (w->shared_up && (w->shared_inter <= 0 || w->shared_inter % 128 || w->hidden % 128 || !aligned(w->shared_up, 16) || !aligned(w->shared_down, 16)))
    return HB_EINVAL;
  return HB_OK;
}

}  // namespace

int hb::nvfp4_tune(const char* key, int value) {
  std::atomic<int>* slot = !strcmp(key, "nvfp4_tile") ? &g_nvfp4_tile : !strcmp(key, "nvfp4_ksplit") ? &g_nvfp4_ksplit : !strcmp(key, "nvfp4_nbw") ? &g_nvfp4_nbw
              : !strcmp(key, "nvfp4_few") ? &g_nvfp4_few : !strcmp(key, "nvfp4_tile_ks") ? &g_nvfp4_tile_ks
              : !strcmp(key, "nvfp4_lag") ? &g_nvfp4_lag : !strcmp(key, "nvfp4_fused") ? &g_nvfp4_fused : nullptr;
  if (!slot || value < 0 || value > 16) return HB_EINVAL;
  *slot = value;
  return HB_OK;
}

extern "C" size_t hb_nvfp4_moe_workspace_bytes(int m, int topk, const hb_nvfp4_experts* routed) {
  if (!routed || m <= 0 || topk <= 0 || check_experts(routed) != HB_OK) return 0;
  return moe_carve(nullptr, m, topk, routed->experts, routed->inter, routed->hidden_out, 0).bytes;
}

extern "C" int hb_nvfp4_moe(const hb_nvfp4_experts* routed, const void* x, const int32_t* ids, const float* weights, int m, int topk, int mode,
                            void* out, void* workspace, size_t workspace_bytes, void* stream) {
  return hb_nvfp4_moe_among(routed, 0, x, ids, weights, m, topk, mode, out, workspace, workspace_bytes, stream);
}

extern "C" int hb_nvfp4_moe_among(const hb_nvfp4_experts* routed, int experts_total, const void* x, const int32_t* ids, const float* weights, int m,
                                  int topk, int mode, void* out, void* workspace, size_t workspace_bytes, void* stream) {
  if (int e = check_experts(routed)) return e;
  if (!x || !ids || !weights || !out || !workspace) return HB_ENULL;
  if (m <= 0 || topk <= 0 || mode < HB_MOE_SUM || mode > HB_MOE_PAIRS_BF16) return HB_EINVAL;
  if (!aligned(x, 16) || !aligned(ids, 4) || !aligned(weights, 4) || !aligned(out, 8) || !aligned(workspace, 16)) return HB_EINVAL;
  const MoeWorkspace ws = moe_carve(workspace, m, topk, routed->experts, routed->inter, routed->hidden_out, 0);
  if (workspace_bytes < ws.bytes) return HB_EWORKSPACE;
  const bool sum = mode == HB_MOE_SUM;
  void* pairs_out = sum ? static_cast<void*>(ws.y) : out;
  // a summed prefill-sized call keeps its pair outputs in BF16: half the traffic of its widest tensor, as the reference's
  // layer does from the same size (hibana/model/flashnext/moe.py:186)
  const bool narrow = sum && m >= MOE_WIDE_ROWS;
  if (int e = run_experts(routed, x, ids, m, topk, ws, pairs_out, mode == HB_MOE_PAIRS_BF16 || narrow, as_stream(stream), experts_total)) return e;
  if (sum) {
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
    moe_launch_combine(c, as_stream(stream));
  }
  return launch_status();
}

extern "C" size_t hb_latent_workspace_bytes(const hb_latent_weights* w, int m, int topk) {
  if (check_latent(w, m, topk) != HB_OK) return 0;
  return latent_carve(w, nullptr, m, topk).bytes;
}

static LatentRouter latent_router_of(const hb_latent_weights* w, const void* x, int m, int topk, const int32_t* slots, int steps, int pad_id, float* fused,
                                     int32_t* ids, float* weights, void* lat, const LatentWorkspace& l) {
  LatentRouter r{};
  r.w = static_cast<const uint16_t*>(w->gate_fc1);
  r.bias = w->bias;
  r.x = static_cast<const uint16_t*>(x);
  r.slots = slots;
  r.m = m;
  r.experts = w->experts_total;
  r.latent = w->latent;
  r.hidden = w->hidden;
  r.topk = topk;
  r.steps = steps;
  r.pad_id = pad_id;
  r.fused = fused;
  r.ids = ids;
  r.weights = weights;
  r.lat = static_cast<uint16_t*>(lat);
  if (w->routed) {
    r.e_lo = w->routed->base;
    r.e_n = w->routed->experts;
    r.ws = &l.moe;
  }
  return r;
}

extern "C" int hb_latent_router(const hb_latent_weights* w, const void* x, int m, int topk, const int32_t* slots, int steps, int route, int pad_id,
                                float* fused, int32_t* ids, float* weights, void* lat, void* workspace, size_t workspace_bytes, void* stream) {
  if (int e = check_latent(w, m, topk)) return e;
  if (!x || !fused || !lat || !workspace || (route && (!ids || !weights))) return HB_ENULL;
  if (!aligned(x, 16) || !aligned(fused, 4) || !aligned(ids, 4) || !aligned(weights, 4) || !aligned(lat, 2) || !aligned(slots, 4) || !aligned(workspace, 16))
    return HB_EINVAL;
  if (pad_id > w->experts_total || steps <= 0) return HB_EINVAL;
  if (int e = moe_check_route(m, w->experts_total, topk)) return e;
  const LatentWorkspace l = latent_carve(w, workspace, m, topk);
  if (workspace_bytes < l.bytes) return HB_EWORKSPACE;
  const LatentRouter r = latent_router_of(w, x, m, topk, slots, steps, pad_id, fused, ids, weights, lat, l);
  if (int e = launch_front(r, as_stream(stream))) return e;
  if (route)
    if (int e = latent_launch_route(r, as_stream(stream))) return e;
  return launch_status();
}

extern "C" int hb_latent_shared_up(const hb_latent_weights* w, const void* x, int m, int topk, void* workspace, size_t workspace_bytes, void* stream) {
  if (int e = check_latent(w, m, topk)) return e;
  if (!x || !workspace || !w->shared_up) return HB_ENULL;
  if (!aligned(x, 16) || !aligned(workspace, 16)) return HB_EINVAL;
  const LatentWorkspace l = latent_carve(w, workspace, m, topk);
  if (workspace_bytes < l.bytes) return HB_EWORKSPACE;
  StreamParams up = dense_params(w->shared_up, w->shared_up_scale, w->shared_inter, w->hidden, x, m, l.shared_h);
  if (int e = launch_nvfp4<EPI_DENSE_RELU2>(up, 1, 1, as_stream(stream))) return e;
  return launch_status();
}

extern "C" int hb_latent_out(const hb_latent_weights* w, const void* routed, int m, int topk, void* out, void* workspace, size_t workspace_bytes,
                             void* stream) {
  if (int e = check_latent(w, m, topk)) return e;
  if (!routed || !out || !workspace) return HB_ENULL;
  if (!aligned(routed, 16) || !aligned(out, 2) || !aligned(workspace, 16)) return HB_EINVAL;
  const LatentWorkspace l = latent_carve(w, workspace, m, topk);
  if (workspace_bytes < l.bytes) return HB_EWORKSPACE;
  if (w->shared_up) {  // the shared expert's down projection of what hb_latent_shared_up left
    StreamParams down = dense_params(w->shared_down, w->shared_down_scale, w->hidden, w->shared_inter, l.shared_h, m, l.shared_y);
    if (int e = launch_nvfp4<EPI_DENSE>(down, 1, 1, as_stream(stream))) return e;
  }
  if (int e = latent_launch_out(static_cast<const uint16_t*>(w->fc2), static_cast<const uint16_t*>(routed), w->shared_up ? l.shared_y : nullptr,
                                static_cast<uint16_t*>(out), m, w->hidden, w->latent, as_stream(stream)))
    return e;
  return launch_status();
}

// The end of a latent block: the routed rows' sums, then out = bf16(shared + sum fc2^T).
static int latent_finish(const hb_latent_weights* w, const int32_t* ids, const float* weights, int m, int topk, const LatentWorkspace& l, void* out, hipStream_t s) {
  CombineParams c{};
  c.pairs = l.moe.y;
  c.ids = ids;
  c.weights = weights;
  c.e_lo = w->routed->base;
  c.e_n = w->routed->experts;
  c.m = m;
  c.topk = topk;
  c.h = w->latent;
  c.out = l.routed;
  moe_launch_combine(c, s);
  if (int e = latent_launch_out(static_cast<const uint16_t*>(w->fc2), l.routed, w->shared_up ? l.shared_y : nullptr, static_cast<uint16_t*>(out), m, w->hidden,
                                w->latent, s))
    return e;
  return launch_status();
}

extern "C" int hb_latent_block(const hb_latent_weights* w, const void* x, const void* lat, const int32_t* ids, const float* weights, int m, int topk,
                               int plan, void* out, void* workspace, size_t workspace_bytes, void* stream) {
  if (int e = check_latent(w, m, topk)) return e;
  if (!w->routed) return HB_ENULL;
  if (!x || !lat || !ids || !weights || !out || !workspace) return HB_ENULL;
  if (!aligned(x, 16) || !aligned(lat, 16) || !aligned(ids, 4) || !aligned(weights, 4) || !aligned(out, 2) || !aligned(workspace, 16)) return HB_EINVAL;
  const LatentWorkspace l = latent_carve(w, workspace, m, topk);
  if (workspace_bytes < l.bytes) return HB_EWORKSPACE;
  const hb_nvfp4_experts* ex = w->routed;
  hipStream_t s = as_stream(stream);
  const int64_t pairs = (int64_t)m * topk, slots = moe_max_slots(pairs, ex->experts, 0, ROWS_PER_SLOT), est = busy_slots(pairs, ex->experts, slots);
  if (plan)
    if (int e = moe_launch_plan(ids, pairs, ex->base, ex->experts, 0, l.moe, s)) return e;
  StreamParams fc1, fc2;
  expert_params(ex, lat, m, topk, l.moe, l.moe.y, 0, fc1, fc2);
  if (w->shared_up) {
    StreamParams up = dense_params(w->shared_up, w->shared_up_scale, w->shared_inter, w->hidden, x, m, l.shared_h);
    StreamParams down = dense_params(w->shared_down, w->shared_down_scale, w->hidden, w->shared_inter, l.shared_h, m, l.shared_y);
    if (int e = ex->gated ? launch_twin<EPI_FC1_GATED, EPI_DENSE_RELU2>(fc1, slots, est, up, 1, s) : launch_twin<EPI_FC1_RELU2, EPI_DENSE_RELU2>(fc1, slots, est, up, 1, s))
      return e;
    if (int e = launch_twin<EPI_FC2, EPI_DENSE>(fc2, slots, est, down, 1, s)) return e;
  } else {
    if (int e = ex->gated ? launch_nvfp4<EPI_FC1_GATED>(fc1, slots, est, s) : launch_nvfp4<EPI_FC1_RELU2>(fc1, slots, est, s)) return e;
    if (int e = launch_nvfp4<EPI_FC2>(fc2, slots, est, s)) return e;
  }
  return latent_finish(w, ids, weights, m, topk, l, out, s);
}

// The block from its rows in one call: [workspace of the router and the block][latent rows][router product][ids][weights].
namespace {
struct LatentLayer {
  LatentWorkspace l;
  uint16_t* lat;
  float* fused;
  int32_t* ids;
  float* weights;
  size_t bytes;
};
LatentLayer latent_layer_carve(const hb_latent_weights* w, void* base, int m, int topk) {
  LatentLayer c{latent_carve(w, base, m, topk), nullptr, nullptr, nullptr, nullptr, 0};
  size_t off = c.l.bytes;
  auto take = [&](size_t bytes) {
    void* ptr = base ? static_cast<char*>(base) + off : nullptr;
    off += (bytes + 255) & ~(size_t)255;
    return ptr;
  };
  c.lat = static_cast<uint16_t*>(take((size_t)m * w->latent * 2));
  c.fused = static_cast<float*>(take((size_t)m * (w->experts_total + w->latent) * 4));
  c.ids = static_cast<int32_t*>(take((size_t)m * topk * 4));
  c.weights = static_cast<float*>(take((size_t)m * topk * 4));
  c.bytes = off;
  return c;
}
}  // namespace

extern "C" size_t hb_latent_layer_workspace_bytes(const hb_latent_weights* w, int m, int topk) {
  if (check_latent(w, m, topk) != HB_OK || !w->routed) return 0;
  return latent_layer_carve(w, nullptr, m, topk).bytes;
}

extern "C" int hb_latent_layer(const hb_latent_weights* w, const void* x, int m, int topk, const int32_t* slots, int steps, int pad_id, void* out,
                               void* workspace, size_t workspace_bytes, void* stream) {
  if (int e = check_latent(w, m, topk)) return e;
  if (!w->routed || !x || !out || !workspace) return HB_ENULL;
  if (!aligned(x, 16) || !aligned(slots, 4) || !aligned(out, 2) || !aligned(workspace, 16)) return HB_EINVAL;
  if (pad_id > w->experts_total || steps <= 0) return HB_EINVAL;
  if (int e = moe_check_route(m, w->experts_total, topk)) return e;
  const LatentLayer c = latent_layer_carve(w, workspace, m, topk);
  if (workspace_bytes < c.bytes) return HB_EWORKSPACE;
  const LatentWorkspace& l = c.l;
  const hb_nvfp4_experts* ex = w->routed;
  hipStream_t s = as_stream(stream);
  const LatentRouter r = latent_router_of(w, x, m, topk, slots, steps, pad_id, c.fused, c.ids, c.weights, c.lat, l);
  StreamParams up, down, fc1, fc2;
  if (w->shared_up) {
    up = dense_params(w->shared_up, w->shared_up_scale, w->shared_inter, w->hidden, x, m, l.shared_h);
    down = dense_params(w->shared_down, w->shared_down_scale, w->hidden, w->shared_inter, l.shared_h, m, l.shared_y);
  }
  const int64_t pairs = (int64_t)m * topk, slot_cap = moe_max_slots(pairs, ex->experts, 0, ROWS_PER_SLOT), est = busy_slots(pairs, ex->experts, slot_cap);
  expert_params(ex, c.lat, m, topk, l.moe, l.moe.y, 0, fc1, fc2);
  if (int e = shape_nvfp4(fc1, est)) return e;
  if (int e = launch_front(r, s)) return e;
  LatentPlan q;
  // Up beside routing and plan, else beside fc1, where more than eight rows take it longer than those two (its splits of K are fc1's launch's, of more than twelve
  // chunks here): the block of 512 experts (1024, 2688) and a shared one of 5376, K split two ways, beside the plan (25.4 us) and so: nine rows 125 and 125, twelve
  // 147 and 143, sixteen 172 and 165; eight rows, four ways, 104 and 110; 512 (512, 2688) and 2048, two ways, four rows 56.6 and 58.7, eight 75.1 and 76.0.
  bool planned = w->shared_up != nullptr;
  if (planned) {
    if (int e = shape_beside(up, 1, fc1)) return e;
    planned = (m <= FP4_FEW_ROWS || up.chunks <= 12 * up.ks) && latent_plan_of(r, q);
  }
  if (int e = planned ? launch_latent_plan(r, q, up, fc1, s) : latent_launch_route(r, s)) return e;
  StreamParams* dense = w->shared_up ? &down : nullptr;
  const bool together = planned == (dense != nullptr) && fc12_serves(pairs, ex->experts, experts_named(w->experts_total, ex->base, ex->experts), fc1, fc2) &&
                        (ex->gated ? launch_fc12<EPI_FC1_GATED>(fc1, fc2, slot_cap, est, dense, s) : launch_fc12<EPI_FC1_RELU2>(fc1, fc2, slot_cap, est, dense, s)) == HB_OK;
  if (!together) {
    if (dense && !planned) {
      if (int e = ex->gated ? launch_twin<EPI_FC1_GATED, EPI_DENSE_RELU2>(fc1, slot_cap, est, up, 1, s) : launch_twin<EPI_FC1_RELU2, EPI_DENSE_RELU2>(fc1, slot_cap, est, up, 1, s))
        return e;
    } else {
      if (int e = ex->gated ? launch_nvfp4<EPI_FC1_GATED>(fc1, slot_cap, est, s) : launch_nvfp4<EPI_FC1_RELU2>(fc1, slot_cap, est, s)) return e;
    }
    if (int e = dense ? launch_twin<EPI_FC2, EPI_DENSE>(fc2, slot_cap, est, down, 1, s) : launch_nvfp4<EPI_FC2>(fc2, slot_cap, est, s)) return e;
  }
  return latent_finish(w, c.ids, c.weights, m, topk, l, out, s);
}
