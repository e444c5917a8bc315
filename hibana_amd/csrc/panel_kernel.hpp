// Dense contractions against packed weights on the matrix cores, shared by the weight formats: a slot of up to 128
// activation rows against `nbw` neighbouring 64-row weight blocks, K split `ks` ways among the wavefronts of ONE workgroup.
//
// A wavefront owns a 64-row block over its split of K and 16 MT activation rows: MT x 4 accumulator tiles. It expands each
// weight once, in registers (Fmt::fragment: scaled BF16, exact), and uses it for MT products. The activations of a
// half chunk (64 k) lie in LDS, one copy a split, shared by the split's nbw wavefronts: brought by LDS-direct loads as 1 KB
// pieces of eight rows x 128 contiguous bytes (reading fragments straight from the L2 instead, sixteen rows x 64 bytes a load,
// runs at 11 B/clk a compute unit: 65 us against 32 at 77 rows, 25600 x 5120), two buffers, a barrier a half chunk. The
// weights of the next chunk wait in a slot of LDS of the wavefront's own.
//
// What bounds it is the issue port and the matrix core together: a product holds the core for 16 cycles and the port for
// about 7, a vector instruction the port for 4.6, and a fragment (eight weights a lane) costs 17 (NVFP4) to 24 (W3) of them.
// So the expansion of the NEXT fragment stands between the products of this one, an instruction or a few behind each
// (two wavefronts a SIMD with two vector instructions a product run at the matrix core's full rate; the same work in
// phases at 88 % of it). A fragment of activations is asked for again, for the next 32-k step, as soon as its last product
// is issued (one set of registers), and the barrier of a half chunk stands after the first quarter of that half's LAST
// step, when its fragments are in registers anyway: the next half's first ones are asked for beside the rest of it.
#pragma once

#include <algorithm>

#include "ring.hpp"
#include "stream_common.hpp"

namespace hb {

constexpr int PANEL_HALF = 64;       // k of a half chunk
constexpr int PANEL_WAVES = 8;       // at most, a workgroup
constexpr int PANEL_LDS = 160 * 1024;
constexpr int PANEL_MT = 8;          // row tiles of a dense call's slot, at most

// The fewest blocks of a workgroup. A split's half chunk of activations is 2 mt pieces, brought by the split's wavefronts, one a
// block, each of which holds its pieces' addresses in registers: eight at most, and four at seven and eight row tiles (five at a routed
// slot's nine), where the accumulators take most of them. (Whether a cut fits the LDS is panel_lds_bytes' to say.)
constexpr int panel_least_blocks(int mt) { return mt <= 4 ? 1 : mt <= 6 ? 2 : 4; }

// A workgroup's part of the launch: its run of blocks, and where several workgroups share a tile's K (kz > 1), which
// share is its own and the tile's number among those.
struct PanelShare {
  int group, z, kz, shared_tile;
};
// A wavefront's: its block of the run, its split and the chunks c0 .. c0 + chunks - 1 of it, and the most chunks a split of
// the workgroup has.
struct PanelWave {
  int ks, nbi, c0, chunks, most;
};
__device__ __forceinline__ PanelWave panel_wave(const StreamParams& p, const PanelShare& part, int wave) {
  PanelWave w;
  w.nbi = (wave * p.ks_inv) >> 16;
  w.ks = wave - w.nbi * p.ks;
  const int z0 = part.kz > 1 ? part.z * p.chunks / part.kz : 0, z1 = part.kz > 1 ? (part.z + 1) * p.chunks / part.kz : p.chunks;
  const int base = ((z1 - z0) * p.ks_inv) >> 16, rem = z1 - z0 - base * p.ks;  // p.ks is a power of two: ks_inv is exact
  w.c0 = z0 + w.ks * base + min(w.ks, rem);
  w.chunks = base + (w.ks < rem ? 1 : 0);
  w.most = base + (rem ? 1 : 0);
  return w;
}

// Sixteen bytes a lane past the caches. The wait state behind the store is its own: a vector instruction right after it may
// overwrite the data registers before the last lanes are read, and the compiler, which guards its own stores, does not know
// this statement for one.
template <class T>
__device__ __forceinline__ void store_through16(T* at, const T& v) { asm volatile("global_store_dwordx4 %0, %1, off sc1\n\ts_nop 1" ::"v"(at), "v"(v) : "memory"); }
template <int N>
__device__ __forceinline__ void wait_vm(void) { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }
__device__ __forceinline__ void wait_lds(void) { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }
template <class T>
__device__ __forceinline__ void pin(T& v) { asm volatile("" : "+v"(v)); }
template <int OFFSET>
__device__ __forceinline__ void ask_lds(u32x4_t& v, uint32_t at) { asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(v) : "v"(at), "n"(OFFSET) : "memory"); }

// acc += w a^T, in place (the builtin lets the compiler move an accumulator to other registers at every product, a third
// more of them in all). The statement hides a matrix instruction from the compiler's wait-state bookkeeping: AFTER_VALU
// stands where the operand w may have been written by the vector instruction before it (two wait states), and products_done
// between the last product and the first other use of an accumulator.
template <bool AFTER_VALU>
__device__ __forceinline__ void product(f32x4_t& acc, const u32x4_t& w, const u32x4_t& a) {
  if constexpr (AFTER_VALU) {
    asm volatile("s_nop 1\n\tv_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+v"(acc) : "v"(w), "v"(a));
  } else {
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+v"(acc) : "v"(w), "v"(a));
  }
}
// ... and behind it the expansion of one pair of weights: convert (two values of the packed dword `from`), times the scale,
// rounded (exactly) into a BF16 pair. One statement, because the compiler guards the seams between its own instructions and
// ours with a wait state each; the two FP32 values live in v64, v65, which a statement cannot name otherwise.
#define HB_PANEL_PAIR(CONVERT, SELECT) CONVERT " v[64:65], %3, 1.0" SELECT "\n\tv_mul_f32 v64, v64, %4\n\tv_mul_f32 v65, v65, %4\n\tv_cvt_pk_bf16_f32 %1, v64, v65"
#define HB_PANEL_PRODUCT_PAIR(NOP, CONVERT, SELECT, acc, out, w, from, scale, a)                                                          \
  asm volatile(NOP "v_mfma_f32_16x16x32_bf16 %0, %2, %5, %0\n\t" HB_PANEL_PAIR(CONVERT, SELECT)                                           \
               : "+v"(acc), "=&v"(out)                                                                                                   \
               : "v"(w), "v"(from), "v"(scale), "v"(a)                                                                                   \
               : "v64", "v65")
#define HB_PANEL_PAIR_ALONE(CONVERT, SELECT, out, from, scale) \
  asm volatile(CONVERT " v[64:65], %1, 1.0" SELECT "\n\tv_mul_f32 v64, v64, %2\n\tv_mul_f32 v65, v65, %2\n\tv_cvt_pk_bf16_f32 %0, v64, v65" : "=&v"(out) : "v"(from), "v"(scale) : "v64", "v65")
// The same in two halves, behind a product each: convert and the first value's scale, then the second's and the rounding.
// `two`: what is between them, bound to the fixed registers.
#define HB_PANEL_PRODUCT_FIRST(NOP, CONVERT, SELECT, acc, two, w, from, scale, a)                            \
  asm volatile(NOP "v_mfma_f32_16x16x32_bf16 %0, %2, %5, %0\n\t" CONVERT " v[64:65], %3, 1.0" SELECT "\n\tv_mul_f32 v64, v64, %4" \
               : "+v"(acc), "=&{v[64:65]}"(two)                                                              \
               : "v"(w), "v"(from), "v"(scale), "v"(a))
typedef __attribute__((ext_vector_type(2))) float panel_two_t;
__device__ __forceinline__ void product_second(f32x4_t& acc, const u32x4_t& w, const u32x4_t& a, panel_two_t& two, float scale, uint32_t& out) {
  asm volatile("v_mfma_f32_16x16x32_bf16 %0, %3, %5, %0\n\tv_mul_f32 v65, v65, %4\n\tv_cvt_pk_bf16_f32 %2, v64, v65"
               : "+v"(acc), "+{v[64:65]}"(two), "=&v"(out)
               : "v"(w), "v"(scale), "v"(a));
}
__device__ __forceinline__ void products_done(void) { asm volatile("s_nop 15\n\ts_nop 7" ::: "memory"); }

// THROUGH: the results are read by other workgroups of the same launch.
template <class Fmt, int EPI, int MT, bool THROUGH = false>
struct Panel {
  typedef typename Fmt::Ring Ring;
  typedef typename Fmt::Chunk Chunk;
  static constexpr int BUF = MT * 16 * PANEL_HALF * 2;  // bytes of one split's half chunk of activations
  static constexpr int PIECES = MT * 2;                 // its 1 KB pieces ...
  static constexpr int HELD = (PIECES + panel_least_blocks(MT) - 1) / panel_least_blocks(MT);  // ... those a wavefront brings at most

  f32x4_t acc[MT][4];
  u32x4_t now[MT];  // the activations' fragments of the step in hand

  // From this many row tiles the products and not the expansion bound a fragment, and a product hides two vector instructions
  // beside it but not four: the pairs are dealt out in halves. Two wavefronts a SIMD, cycles a fragment (the products alone 16
  // each): eight tiles 150.8 with whole pairs and 136.5 with halves, seven 136.7 and 128.8, six 125.1 and 120.5, five 113.9 and 122.1.
  static constexpr int HALVES_FROM = 6;

  // The products of fragment J = 4 * step + tile of a chunk, and between them the expansion of fragment J + 1, a pair of
  // its values behind every MT / 4 products (or half a pair behind every MT / 8; the last of nine
  // has none). The empty statements hold that order: left to itself the compiler puts the expansion behind the products (fewer registers), where nothing runs beside it.
  // FRESH: the activations' fragments may still be on their way (asked for in order, nothing behind them). NEXT >= 0: the
  // LDS offset of the next step's, from `at`.
  template <int J, bool FRESH, int NEXT>
  __device__ __forceinline__ bf16x8_t group(const Chunk& ch, const Slot& sl, bf16x8_t b, uint32_t at) {
    u32x4_t w = __builtin_bit_cast(u32x4_t, b);
    typename Fmt::Part part;
    uint32_t out[4] = {0u, 0u, 0u, 0u};
    panel_two_t two = {0.f, 0.f};
    products<J, FRESH, NEXT, 0>(ch, sl, w, at, part, out, two);
    return __builtin_bit_cast(bf16x8_t, u32x4_t{out[0], out[1], out[2], out[3]});
  }
  template <int J, bool FRESH, int NEXT, int T>
  __device__ __forceinline__ void products(const Chunk& ch, const Slot& sl, u32x4_t& w, uint32_t at, typename Fmt::Part& part, uint32_t (&out)[4],
                                           panel_two_t& two) {
    constexpr int NT = J & 3;
    if constexpr (T < MT) {
      if constexpr (FRESH) {
        asm volatile("s_waitcnt lgkmcnt(%0)" ::"n"(MT - 1 - T) : "memory");
        pin(now[T]);
      }
      if constexpr (J < 15 && T == 0) part = Fmt::template open<((J + 1) & 3), ((J + 1) >> 2)>(ch, sl);
      if constexpr (MT >= HALVES_FROM) {  // halves of pairs: half I goes behind product I MT / 8
        constexpr int I = (8 * T + MT - 1) / MT;
        static_assert(I == 8 || I * MT / 8 == T, "a half for every product, up to the eighth");
        if constexpr (J >= 15 || I == 8) {
          product<T == 0>(acc[T][NT], w, now[T]);
        } else if constexpr (I & 1) {
          product_second(acc[T][NT], w, now[T], two, part.scale, out[I >> 1]);
        } else if constexpr ((I + 1) * MT / 8 == T) {
          Fmt::template product_pair<(I >> 1), T == 0>(acc[T][NT], w, now[T], part, out[I >> 1]);
        } else {
          Fmt::template product_first<(I >> 1), T == 0>(acc[T][NT], w, now[T], part, two);
        }
      } else {
        constexpr int K = (4 * T + MT - 1) / MT;  // the pairs are dealt out evenly: pair K goes behind product K MT / 4
        constexpr bool FIRST = J < 15 && K < 4 && K * MT / 4 == T;
        if constexpr (FIRST) {
          Fmt::template product_pair<K, T == 0>(acc[T][NT], w, now[T], part, out[K]);
        } else {
          product<T == 0>(acc[T][NT], w, now[T]);
        }
        if constexpr (FIRST && K + 1 < 4 && (K + 1) * MT / 4 == T) Fmt::template pair_alone<(K + 1) & 3>(part, out[(K + 1) & 3]);
        if constexpr (FIRST && MT == 1) {
          Fmt::template pair_alone<2>(part, out[2]);
          Fmt::template pair_alone<3>(part, out[3]);
        }
      }
      if constexpr (NEXT >= 0) ask_lds<NEXT + T * 2048>(now[T], at);
      products<J, FRESH, NEXT, T + 1>(ch, sl, w, at, part, out, two);
    }
  }
  static __device__ __forceinline__ bf16x8_t whole(const Chunk& ch, const Slot& sl) {  // fragment 0 of a chunk
    typename Fmt::Part part = Fmt::template open<0, 0>(ch, sl);
    uint32_t out[4];
    Fmt::template pair_alone<0>(part, out[0]);
    Fmt::template pair_alone<1>(part, out[1]);
    Fmt::template pair_alone<2>(part, out[2]);
    Fmt::template pair_alone<3>(part, out[3]);
    return __builtin_bit_cast(bf16x8_t, u32x4_t{out[0], out[1], out[2], out[3]});
  }

  template <int T = 0>
  __device__ __forceinline__ void ask_first(uint32_t at) {
    if constexpr (T < MT) {
      ask_lds<T * 2048>(now[T], at);
      ask_first<T + 1>(at);
    }
  }

  __device__ __forceinline__ void run(const StreamParams& p, const Slot& sl, uint8_t* lds, const PanelShare& part) {
    NoWait none;
    run(p, sl, lds, part, none);
  }
  // `wait`: for the activations, behind the requests of the first weights.
  template <class Wait>
  __device__ __forceinline__ void run(const StreamParams& p, const Slot& sl, uint8_t* lds, const PanelShare& part, Wait& wait) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), q = lane >> 4, r16 = lane & 15;
    const PanelWave share = panel_wave(p, part, wave);
    const int nb = part.group * p.nbw + share.nbi;
    const bool active = nb < p.n_blocks;
    const int mine = 2 * share.chunks, halves = 2 * share.most;  // this split's half chunks; the longest split's, which all wavefronts walk
    uint8_t* abuf = lds + share.ks * 2 * BUF;
    uint8_t* slot = lds + p.ks * 2 * BUF + wave * Fmt::BLOCK_BYTES;
#pragma unroll
    for (int t = 0; t < MT; t++)
#pragma unroll
      for (int nt = 0; nt < 4; nt++) acc[t][nt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    RingSource w;
    w.row = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(sl.w + (int64_t)(active ? nb : 0) * p.chunks * Fmt::BLOCK_BYTES), 0, p.chunks * Fmt::BLOCK_BYTES, 0x00020000);
    uint32_t codes, scales;
    Ring::lanes(w, lane, r16, (uint32_t)(uintptr_t)(lds_ptr_t)slot, codes, scales);
    wait.look();
    Ring::request(w, share.c0, (lds_ptr_t)slot);
    // The split's pieces, dealt to its wavefronts in turn: piece j is rows 8 j .. 8 j + 7, lane l lands at its byte 16 l, the
    // 16-byte column (l & 7) of row 8 j + l / 8 - which holds the row's column (l & 7) ^ (row / 2 & 7), so that the sixteen
    // rows of a fragment read lie in sixteen different 16-byte columns of the LDS.
    const __amdgpu_buffer_rsrc_t arow = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(p.a), 0, (int)p.a_bytes, 0x00020000);
    uint32_t piece[HELD];
#pragma unroll
    for (int j = 0; j < HELD; j++) {
      const int id = j * p.nbw + share.nbi;
      if (id < PIECES) {
        const int row = 8 * id + (lane >> 3);
        piece[j] = (uint32_t)(activation_row_index<EPI>(p, sl, row) * p.a_stride) * 2 + (uint32_t)(((lane & 7) ^ ((row >> 1) & 7)) << 4);
      }
    }
    auto bring = [&](int h) {
#pragma unroll
      for (int j = 0; j < HELD; j++) {
        const int id = j * p.nbw + share.nbi;
        if (id < PIECES)
          __builtin_amdgcn_raw_ptr_buffer_load_lds(arow, (lds_ptr_t)(abuf + (h & 1) * BUF + id * 1024), 16, piece[j], (uint32_t)(share.c0 * 256 + h * (PANEL_HALF * 2)), 0, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    };
    const uint32_t at0 = (uint32_t)(uintptr_t)(lds_ptr_t)abuf + r16 * 128 + ((q ^ (r16 >> 1)) << 4), at1 = at0 ^ 64;
    if (!wait.done()) return;  // nothing is computed or stored
    bring(0);
    bring(1);
    wait_vm<0>();
    __builtin_amdgcn_s_barrier();
    Chunk ch;
    Ring::ask(ch, codes, scales);
    ask_first(at0);
    wait_lds();
    Ring::have(ch);
    if (mine > 2) Ring::request(w, share.c0 + 1, (lds_ptr_t)slot);
    for (int h = 0; h < halves; h += 2) {
      if (h < mine) {
        bf16x8_t b = whole(ch, sl);
        b = group<0, true, -1>(ch, sl, b, 0);
        b = group<1, false, -1>(ch, sl, b, 0);
        b = group<2, false, -1>(ch, sl, b, 0);
        b = group<3, false, 0>(ch, sl, b, at1);
        b = group<4, true, -1>(ch, sl, b, 0);
        if (h + 2 < mine) wait_vm<Ring::LOADS>(); else wait_vm<0>();  // the half after this one has landed; what was asked for behind it are the next weights
        __builtin_amdgcn_s_barrier();
        if (h + 2 < mine) bring(h + 2);
        b = group<5, false, -1>(ch, sl, b, 0);
        b = group<6, false, -1>(ch, sl, b, 0);
        b = group<7, false, BUF>(ch, sl, b, at0);
        b = group<8, true, -1>(ch, sl, b, 0);
        b = group<9, false, -1>(ch, sl, b, 0);
        b = group<10, false, -1>(ch, sl, b, 0);
        b = group<11, false, BUF>(ch, sl, b, at1);
        b = group<12, true, -1>(ch, sl, b, 0);
        wait_vm<0>();
        __builtin_amdgcn_s_barrier();
        if (h + 3 < mine) bring(h + 3);
        b = group<13, false, -1>(ch, sl, b, 0);
        b = group<14, false, -1>(ch, sl, b, 0);
        Chunk after;
        Ring::ask(after, codes, scales);
        group<15, false, 0>(ch, sl, b, at0);
        asm volatile("s_waitcnt lgkmcnt(%0)" ::"n"(MT) : "memory");  // the weights; the fragments' own waits follow
        Ring::have(after);
        ch = after;
        if (h + 4 < mine) Ring::request(w, share.c0 + (h >> 1) + 2, (lds_ptr_t)slot);
      } else {
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_s_barrier();
      }
    }
    wait_lds();
    products_done();
#pragma unroll
    for (int t = 0; t < MT; t++)
#pragma unroll
      for (int nt = 0; nt < 4; nt++) pin(acc[t][nt]);
    if (p.ks == 1 && part.kz == 1 && !((reinterpret_cast<uintptr_t>(p.out) | (uintptr_t)(p.out_stride * 2)) & 15)) {
      if (active) store_rows(p, sl, slot, nb, lane);
    } else {
      finish(p, sl, lds, part, nb, active, share.ks, share.nbi, lane);
    }
  }

  typedef __attribute__((ext_vector_type(2))) uint32_t u32x2_t;
  static constexpr bool GATED = EPI == EPI_FC1_GATED;
  // The FP32 scales of a lane's output columns: one a column of each 16-row tile, or the matrix's one.
  static __device__ __forceinline__ f32x4_t column_scales(const Slot& sl, int nb, int tile, int q) {
    typedef f32x4_t __attribute__((aligned(4))) loose_f32x4_t;  // row scales start on any float
    return Fmt::PER_ROW ? *reinterpret_cast<const loose_f32x4_t*>(sl.rs + nb * 64 + 16 * tile + 4 * q) : f32x4_t{sl.scalar, sl.scalar, sl.scalar, sl.scalar};
  }
  // Four neighbouring output columns as BF16 (gated: v0 / s0 the up tile, v1 / s1 the gate tile).
  static __device__ __forceinline__ u32x2_t rounded(const f32x4_t& v0, const f32x4_t& v1, const f32x4_t& s0, const f32x4_t& s1) {
    float y[4];
#pragma unroll
    for (int r = 0; r < 4; r++) {
      y[r] = v0[r] * s0[r];
      if (GATED) {
        const uint32_t ug = bf16_pair(y[r], v1[r] * s1[r]);  // up and gate rounded to BF16 ...
        y[r] = silu(pair_hi(ug)) * pair_lo(ug);              // ... and their product, rounded below
      }
    }
    if (EPI == EPI_FC1_RELU2 || EPI == EPI_DENSE_RELU2) {  // bf16(relu(bf16(y))^2), two values a conversion
      const uint32_t u01 = bf16_pair(y[0], y[1]), u23 = bf16_pair(y[2], y[3]);
      // relu on the bits: a negative value (and -0) is a negative integer; a NaN stays one, as torch's relu leaves it
      const float h0 = __int_as_float(max((int)(u01 << 16), 0)), h1 = __int_as_float(max((int)(u01 & 0xffff0000u), 0));
      const float h2 = __int_as_float(max((int)(u23 << 16), 0)), h3 = __int_as_float(max((int)(u23 & 0xffff0000u), 0));
      y[0] = h0 * h0, y[1] = h1 * h1, y[2] = h2 * h2, y[3] = h3 * h3;
    }
    return u32x2_t{bf16_pair(y[0], y[1]), bf16_pair(y[2], y[3])};
  }

  // One lane's four neighbouring output columns of a tile (gated: of pair `nt` of tiles), stored as they are.
  static __device__ __forceinline__ void emit(const StreamParams& p, const Slot& sl, int nb, int t, int nt, int lane, const f32x4_t& v0, const f32x4_t& v1) {
    const int q = lane >> 4, i = 16 * t + (lane & 15);
    if (i >= sl.rows) return;
    const int64_t pos = sl.p0 + i;
    const f32x4_t s0 = column_scales(sl, nb, GATED ? 2 * nt : nt, q), s1 = GATED ? column_scales(sl, nb, 2 * nt + 1, q) : s0;
    const int64_t at = (EPI == EPI_FC2 ? (int64_t)p.order[pos] : pos) * p.out_stride + nb * (GATED ? 32 : 64) + 16 * nt + 4 * q;
    if (EPI != EPI_FC2 || p.out_bf16) {
      const u32x2_t v = rounded(v0, v1, s0, s1);
      u32x2_t* to = reinterpret_cast<u32x2_t*>(reinterpret_cast<uint16_t*>(p.out) + at);
      if constexpr (THROUGH) store_through(reinterpret_cast<uint64_t*>(to), __builtin_bit_cast(uint64_t, v)); else *to = v;
    } else {
      *reinterpret_cast<f32x4_t*>(reinterpret_cast<float*>(p.out) + at) = v0 * s0;
    }
  }

  // All of a wavefront's results where it holds them K-complete, as whole rows: a lane's four columns of sixteen rows are 32
  // bytes a row and store, so a row tile goes through the wavefront's own (by now empty) slot of LDS and leaves as 128 (gated:
  // 64) contiguous bytes a row; what the stores need from memory (the rows' places, the column scales) is asked for once, ahead
  // of the first. Before, the last row tiles of a slot of 128 stood behind eight round trips to `order`: 11.9 us of a workgroup's
  // 23.9 (fc2 of the three-bit layer, 1543 rows), 14.6 of 68.6 (the latent block's, 2048). A row of LDS is 144 bytes: sixteen
  // rows' columns start in different banks.
  static constexpr int LINE = 144;
  static_assert(16 * LINE <= Fmt::BLOCK_BYTES && LINE % 16 == 0 && Fmt::BLOCK_BYTES % 16 == 0, "a row tile in the slot of a weight block");
  __device__ __forceinline__ void store_rows(const StreamParams& p, const Slot& sl, uint8_t* slot, int nb, int lane) {
    constexpr int PER_ROW = GATED ? 4 : 8, ROWS = 64 / PER_ROW, PASSES = 16 / ROWS;  // lanes a row, rows a store, stores a row tile
    const int q = lane >> 4, r16 = lane & 15, line = lane / PER_ROW, part = lane % PER_ROW;
    f32x4_t scale[4];
#pragma unroll
    for (int nt = 0; nt < 4; nt++) scale[nt] = column_scales(sl, nb, nt, q);
    int row[MT * PASSES];
#pragma unroll
    for (int j = 0; j < MT * PASSES; j++) {
      row[j] = sl.p0 + min(ROWS * j + line, sl.rows - 1);
      if (EPI == EPI_FC2) row[j] = p.order[row[j]];
    }
    const bool wide = EPI == EPI_FC2 && !p.out_bf16;  // FP32: two tiles' columns are a row of LDS
    uint8_t* out = static_cast<uint8_t*>(p.out) + (int64_t)nb * (GATED ? 64 : wide ? 256 : 128) + 16 * part;
    const int64_t pitch = p.out_stride * (wide ? 4 : 2);
    uint8_t* write = slot + r16 * LINE;
    const uint8_t* read = slot + line * LINE + 16 * part;
    auto leave = [&](int t, int offset) {
      asm volatile("" ::: "memory");  // the lanes read what other lanes of the wavefront wrote: LDS serves a wavefront in order
#pragma unroll
      for (int u = 0; u < PASSES; u++) {
        const u32x4_t v = *reinterpret_cast<const u32x4_t*>(read + u * ROWS * LINE);
        if (16 * t + ROWS * u + line < sl.rows) {
          u32x4_t* to = reinterpret_cast<u32x4_t*>(out + row[PASSES * t + u] * pitch + offset);
          if constexpr (THROUGH) store_through16(to, v); else *to = v;
        }
      }
      asm volatile("" ::: "memory");
    };
#pragma unroll
    for (int t = 0; t < MT; t++) {
      if (16 * t >= sl.rows) break;
      if (wide) {
#pragma unroll
        for (int nt = 0; nt < 4; nt += 2) {
          *reinterpret_cast<f32x4_t*>(write + 16 * q) = acc[t][nt] * scale[nt];
          *reinterpret_cast<f32x4_t*>(write + 64 + 16 * q) = acc[t][nt + 1] * scale[nt + 1];
          leave(t, 64 * nt);
        }
      } else {
#pragma unroll
        for (int nt = 0; nt < (GATED ? 2 : 4); nt++) {
          const int a = GATED ? 2 * nt : nt, b = GATED ? 2 * nt + 1 : nt;
          *reinterpret_cast<u32x2_t*>(write + 32 * nt + 8 * q) = rounded(acc[t][a], acc[t][b], scale[a], scale[b]);
        }
        leave(t, 0);
      }
    }
  }

  // What becomes of a K-complete (over this workgroup's share) result: stored, or left in memory for the workgroup that
  // arrives last.
  static __device__ __forceinline__ void deliver(const StreamParams& p, const Slot& sl, const PanelShare& part, int nb, int nbi, int t, int nt, int lane, const f32x4_t& v0,
                                                 const f32x4_t& v1) {
    if (part.kz > 1) {
      store_through16(partial_at(p, part, part.z, nbi, t, nt) + lane, v0);
    } else {
      emit(p, sl, nb, t, nt, lane, v0, v1);
    }
  }
  static __device__ __forceinline__ f32x4_t* partial_at(const StreamParams& p, const PanelShare& part, int z, int nbi, int t, int nt) {
    return reinterpret_cast<f32x4_t*>(p.partial) + ((((int64_t)part.shared_tile * part.kz + z) * p.nbw + nbi) * (MT * 4) + t * 4 + nt) * 64;
  }

  // The K splits' tiles meet in LDS, two row tiles at a time, and are added in split order; each split's wavefront takes
  // every ks-th of the results. Where further workgroups share the tile's K, all leave their results in memory (written
  // through and waited for) and draw a ticket; the last one adds them in the order of the shares: the same sum whichever
  // it is. The tickets lie at a fixed place in the workspace and are zero again when the launch ends.
  __device__ __forceinline__ void finish(const StreamParams& p, const Slot& sl, uint8_t* lds, const PanelShare& part, int nb, bool active, int ks, int nbi, int lane) {
    if (p.ks == 1) {
      if (active) {
#pragma unroll
        for (int t = 0; t < MT; t++) {
          if (16 * t < sl.rows) {
#pragma unroll
            for (int nt = 0; nt < (GATED ? 2 : 4); nt++) deliver(p, sl, part, nb, nbi, t, nt, lane, acc[t][GATED ? 2 * nt : nt], acc[t][GATED ? 2 * nt + 1 : nt]);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    } else {
      f32x4_t* all = reinterpret_cast<f32x4_t*>(lds);
      f32x4_t* mine = all + (nbi * p.ks + ks) * 512 + lane;
      const f32x4_t* first = all + nbi * p.ks * 512 + lane;
#pragma unroll
      for (int t0 = 0; t0 < MT; t0 += 2) {
        __syncthreads();  // the memory is free: the last fragments, or the tiles before these, have been read
#pragma unroll
        for (int u = 0; u < 8; u++)
          if (t0 + (u >> 2) < MT) mine[u * 64] = acc[t0 + (u >> 2) < MT ? t0 + (u >> 2) : 0][u & 3];
        __syncthreads();
        if (active) {
          for (int u = ks; u < (GATED ? 4 : 8); u += p.ks) {
            const int t = t0 + (GATED ? u >> 1 : u >> 2), nt = GATED ? u & 1 : u & 3, from = GATED ? 2 * u : u;
            if (t >= MT || 16 * t >= sl.rows) continue;
            f32x4_t v0 = first[from * 64], v1 = v0;
            if (GATED) v1 = first[(from + 1) * 64];
            for (int s = 1; s < p.ks; s++) {
              v0 += first[s * 512 + from * 64];
              if (GATED) v1 += first[s * 512 + (from + 1) * 64];
            }
            deliver(p, sl, part, nb, nbi, t, nt, lane, v0, v1);
          }
        }
      }
    }
    if (GATED || part.kz == 1) return;  // (calls that share K among workgroups are dense)
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wavefront's results are in memory before the count
    __syncthreads();
    int* last = reinterpret_cast<int*>(lds);
    if (threadIdx.x == 0) {
      unsigned int* ticket = p.panel_tickets + part.shared_tile;
      *last = atomicAdd(ticket, 1u) == (unsigned)part.kz - 1u;
      if (*last) *ticket = 0u;
    }
    __syncthreads();
    if (!*last || !active) return;
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");  // drop what this compute die's L2 holds of the others' results
    constexpr int BATCH = 4;  // results whose shares are asked for together, a share ahead of the one being added
    const int count = (MT * 4 - ks + p.ks - 1) / p.ks;  // what this wavefront delivered: results ks, ks + p.ks, ...
    auto unit = [&](int i) { return i * p.ks + ks; };
    for (int i0 = 0; i0 < count; i0 += BATCH) {
      f32x4_t sum[BATCH], more[BATCH];
      auto load = [&](f32x4_t (&to)[BATCH], int z) {
#pragma unroll
        for (int j = 0; j < BATCH; j++) to[j] = partial_at(p, part, z, nbi, 0, unit(min(i0 + j, count - 1)))[lane];
      };
      load(sum, 0);
      load(more, 1);
      for (int z = 1; z < part.kz; z++) {
        f32x4_t then[BATCH];
        if (z + 1 < part.kz) load(then, z + 1);
#pragma unroll
        for (int j = 0; j < BATCH; j++) {
          sum[j] += more[j];
          more[j] = then[j];
        }
      }
#pragma unroll
      for (int j = 0; j < BATCH; j++) {
        const int u = unit(i0 + j);
        if (i0 + j < count && 16 * (u >> 2) < sl.rows) emit(p, sl, nb, u >> 2, u & 3, lane, sum[j], sum[j]);
      }
    }
  }
};

// Dense calls: every slot has up to 16 MT rows. The tiles past p.panel_full have their K shared by p.panel_kz workgroups each.
template <class Fmt, int EPI, int MT>
__global__ __launch_bounds__(64 * PANEL_WAVES, 2) void panel_kernel(StreamParams p) {
  extern __shared__ __align__(128) uint8_t panel_lds[];  // (the addresses of the halves of a row differ in one bit)
  int tile = blockIdx.x;
  PanelShare part{0, 0, 1, 0};
  if (tile >= p.panel_full) {
    const int r = tile - p.panel_full;
    part.shared_tile = r / p.panel_kz;
    part.z = r - part.shared_tile * p.panel_kz;
    part.kz = p.panel_kz;
    tile = p.panel_full + part.shared_tile;
  }
  // Workgroups go to the eight compute dies in turn; a die's take neighbouring runs of blocks, all slots of a run one after
  // the other, so that a run's weights come into one L2 once (25600 x 5120, four matrices in turn: 2048 rows 436 -> 422 us, 512 rows 142 -> 126).
  const int even = p.panel_full & ~7;
  if (tile < even) tile = (tile & 7) * (even >> 3) + (tile >> 3);
  part.group = tile / p.panel_slots;
  const int slot = tile - part.group * p.panel_slots;
  const Slot sl = slot_of<EPI>(p, slot);
  if (sl.rows <= 0) return;
  Panel<Fmt, EPI, MT> panel;
  panel.run(p, sl, panel_lds, part);
}

template <class Fmt>
inline size_t panel_lds_bytes(int mt, int ks, int nbw) {
  const size_t loop = (size_t)ks * 2 * mt * 2048 + (size_t)ks * nbw * Fmt::BLOCK_BYTES, exchange = ks > 1 ? (size_t)ks * nbw * 8192 : 0;
  return loop > exchange ? loop : exchange;
}


template <class Fmt, int EPI, int MT, bool THROUGH, class Wait>  // as many row tiles as the slot's rows need, MT at most (light slots do not come here)
__device__ __forceinline__ void panel_tiles(const StreamParams& p, const Slot& sl, uint8_t* lds, const PanelShare& part, Wait& wait) {
  if constexpr (MT > 1 + Fmt::LIGHT_ROWS / 16) {
    if ((sl.rows + 15) >> 4 < MT) return panel_tiles<Fmt, EPI, MT - 1, THROUGH>(p, sl, lds, part, wait);
  }
  Panel<Fmt, EPI, MT, THROUGH> panel;
  panel.run(p, sl, lds, part, wait);
}
template <class Fmt, int EPI, int MOST, bool THROUGH, class Wait>
__device__ __forceinline__ void panel_slot(const StreamParams& p, const Slot& sl, int group, uint8_t* lds, Wait& wait) {
  const PanelShare part{group, 0, 1, 0};
  if (sl.rows <= Fmt::LIGHT_ROWS) return Fmt::template light<EPI>(p, sl, group, lds, wait);
  panel_tiles<Fmt, EPI, MOST, THROUGH>(p, sl, lds, part, wait);
}

// Routed calls: a plan's slots of up to 16 MOST rows. Workgroups go to the eight compute dies in turn: all of a slot's take
// the same place in that turn, so that its activations come into one L2 once
// (2048 rows, 22 of 512 experts, (1024, 2688): the latent block 811 -> 782 us; 1543 rows of the three-bit layer 285 -> 276).
// A compute unit holds as many workgroups as the registers of the highest slot leave room for: four with slots of 48 rows, three
// with 80, two with 128 and 144 (the choice: panel_height).
template <class Fmt, int EPI, int MOST>
__global__ __launch_bounds__(256, (MOST <= 3 ? 4 : MOST <= 5 ? 3 : 2)) void panel_tile_kernel(StreamParams p) {
  extern __shared__ __align__(128) uint8_t panel_lds[];  // (the addresses of the halves of a row differ in one bit)
  const int die = blockIdx.x & 7, local = blockIdx.x >> 3, round = local / p.panel_groups, slot = 8 * round + die;
  if (slot >= p.panel_full) return;
  const Slot sl = slot_of<EPI>(p, slot);
  if (sl.rows <= 0) return;  // a slot the plan did not fill: the whole workgroup leaves
  NoWait none;
  panel_slot<Fmt, EPI, MOST, false>(p, sl, local - round * p.panel_groups, panel_lds, none);
}

// fc1 and fc2 of a routed call in one launch, as w3_fc12_kernel has them on the stream: fc2's workgroups fill the units that fc1's last
// round leaves idle - where slots are few, a third of the time - and run beside its last ones instead of behind them. A die's workgroups are its slots'
// in fc12_place's order, `lag` of its slots apart. h is written through to memory, and a slot's fc2 workgroups, which ask for their first weights
// ahead of the wait, read it through their die's L2, which holds no older copy of it (a row of h is whole 256-byte pieces). The same sums
// in the same order as the two launches: the same bits. Measured, two launches and one, the whole call, us: three-bit, skewed, 512 experts (2048, 512)
// 1543 rows 231 and 217, 2048 rows 281 and 265, 256 (2560, 768) 1000 rows 247 and 227, 180 (1664, 384) 1000 rows 112 and 98, 64 (2048, 512) 2048 rows 196 and 168; even,
// 128 (1024, 256) 1000 rows 84 and 73; NVFP4, 512 (1024, 2688) 2048 rows of 22 712 and 698, 200 rows 346 and 340, 256 (768, 1536) 500 rows of twelve 136
// and 127, 16 (512, 1024) 40 rows of eight 48 and 46. Where two are the faster: panel_together.
template <class Fmt, int EPI1, int MOST>
__global__ __launch_bounds__(256, (MOST <= 3 ? 4 : MOST <= 5 ? 3 : 2)) void panel_fc12_tile_kernel(StreamParams p1, StreamParams p2, int rounds, int lag) {
  extern __shared__ __align__(128) uint8_t panel_lds[];  // (the addresses of the halves of a row differ in one bit)
  __shared__ int outcome;
  const Fc12Place at = fc12_place(blockIdx.x >> 3, p1.panel_groups, p2.panel_groups, rounds, lag);
  const int slot = 8 * at.slot + (blockIdx.x & 7);
  if (slot >= p1.panel_full) return;
  if (at.is_fc1) {
    const Slot sl = slot_of<EPI1>(p1, slot);
    if (sl.rows <= 0) return;
    NoWait none;
    panel_slot<Fmt, EPI1, MOST, true>(p1, sl, at.index, panel_lds, none);
    fc12_arrive(p1, slot);
  } else {
    const Slot sl = slot_of<EPI_FC2>(p2, slot);
    if (sl.rows <= 0) return;
    SlotWait wait(p2, slot, &outcome, false);
    panel_slot<Fmt, EPI_FC2, MOST, false>(p2, sl, at.index, panel_lds, wait);
  }
}

// How a dense call is cut: row tiles a slot, the shape of a workgroup, the tiles whose K is shared and among how many.
struct PanelPlan {
  int mt, slots, ks, nbw, groups, kz;
  int64_t full, tiles;
  double us;  // the estimate it was chosen by
};
// The tickets of the tiles whose K is shared: a fixed place at the head of the workspace, whatever the call's shape, so that
// no other call's partial results are ever found there; the partial results follow.
constexpr size_t PANEL_TICKET_BYTES = 4096;
constexpr int64_t PANEL_SHARED_TILES = PANEL_TICKET_BYTES / 4 - PLAN_HEADER;
inline size_t panel_room(const PanelPlan& q) { return q.kz > 1 ? PANEL_TICKET_BYTES + (size_t)(q.tiles - q.full) * q.kz * q.nbw * q.mt * 4 * 64 * sizeof(f32x4_t) : 0; }

// The cut with the least estimated time, by a model fitted to 3 300 measured (size, cut) pairs (MI355X, us; 1024 .. 25600
// columns, K 512 .. 5120, 17 .. 2048 rows; the cut it takes is within 2.4 % of the best measured one on average): a chunk of
// a wavefront takes 1.45 + 0.16 mt with two wavefronts a SIMD and 0.7 + 0.1 mt alone; a workgroup's start and end 4.6;
// eight-wavefront workgroups run one a compute unit, four-wavefront ones two where their LDS allows; the last arriver of
// a shared tile reads its partial results at about 46 GB/s and the handing over costs 5.3; all shared tiles' results together
// are written and read at about 2 TB/s (left out, 1024 rows of 25600 x 5120 shared 288 tiles five ways: 318 us, 243
// without). `room`: bytes of the workspace.
template <class Fmt>
inline PanelPlan search_panel(int m, int n_blocks, int chunks, size_t room) {
  static const struct { int ks, nbw; } shapes[] = {{1, 4}, {1, 8}, {2, 2}, {2, 4}, {4, 1}, {4, 2}, {8, 1}};
  PanelPlan best{};
  best.us = 1e30;
  const int least = (m + 127) / 128;
  // A call that fills the device takes the fewest slots its rows allow, or one more (the rows dealt out evenly); a smaller
  // one may be faster in many slots of few row tiles (1024 x 512, 1024 rows: 14.7 us in eight slots, 7.1 in more; 4096 x 1024, 512 rows 18.6 and 10.2).
  const bool small = (int64_t)n_blocks * least <= 512;
  for (int mt = PANEL_MT; mt >= 1; mt--) {
    const int slots = (m + 16 * mt - 1) / (16 * mt);
    if (mt != ((m + least - 1) / least + 15) / 16 && mt != ((m + least) / (least + 1) + 15) / 16 && !(small && slots > least)) continue;
    const double pair = 1.45 + Fmt::EXPAND_US + 0.16 * mt, alone = 0.7 + 0.5 * Fmt::EXPAND_US + 0.105 * mt;
    for (auto& shape : shapes) {
      const size_t lds = panel_lds_bytes<Fmt>(mt, shape.ks, shape.nbw);
      if (lds > PANEL_LDS || shape.nbw < panel_least_blocks(mt) || shape.ks > chunks) continue;
      const bool wide = shape.ks * shape.nbw == 8;
      const int64_t groups = (n_blocks + shape.nbw - 1) / shape.nbw, tiles = groups * ((m + 16 * mt - 1) / (16 * mt));
      const int64_t resident = !wide && 2 * lds <= PANEL_LDS ? 512 : 256;
      auto rounds = [&](int64_t workgroups, int c) {  // us of that many workgroups of c chunks a wavefront
        if (wide && mt <= Fmt::BESIDE_TILES && 2 * lds <= PANEL_LDS && workgroups > 256) return workgroups / 256.0 * (c * pair + 4.6);  // the next ones start beside those at work
        const int64_t whole = workgroups / resident, rest = workgroups - whole * resident;
        const double busy = wide || resident == 512 ? pair : alone;
        return whole * (c * busy + 4.6) + (rest ? c * (wide || rest > 256 ? pair : alone) + 4.6 : 0);
      };
      for (int kz = 1; kz <= 16 && (kz == 1 || chunks / kz >= shape.ks); kz++) {
        const int64_t full = kz == 1 ? tiles : tiles / resident * resident, rest = tiles - full;
        if (kz > 1 && (!rest || rest > PANEL_SHARED_TILES)) continue;
        PanelPlan q{mt, slots, shape.ks, shape.nbw, (int)groups, kz, full, tiles, 0};
        if (panel_room(q) > room) continue;
        q.us = rounds(full, (chunks + shape.ks - 1) / shape.ks);
        const double shared_tile = kz > 1 ? kz * (double)mt * shape.nbw * 4096 : 0;  // bytes of partial results
        if (rest) q.us += rounds(rest * kz, ((chunks + kz - 1) / kz + shape.ks - 1) / shape.ks) + (kz > 1 ? 5.3 + shared_tile / 46e3 + rest * shared_tile / 2e6 : 0);
        if (q.us < best.us * (kz > 1 ? 0.97 : 1.0)) best = q;
      }
    }
  }
  return best;
}

// ... kept for the sizes a thread asks for again and again (the search takes microseconds; the best cut of all and the one
// for a smaller room have places of their own).
constexpr size_t PANEL_ANY_ROOM = ~(size_t)0;
template <class Fmt>
inline const PanelPlan& plan_panel(int m, int n_blocks, int chunks, size_t room) {
  struct Entry {
    int m, n_blocks, chunks;
    size_t room;
    PanelPlan plan;
  };
  static thread_local Entry kept[64];
  Entry& e = kept[((unsigned)m * 31u + (unsigned)n_blocks * 7u + (unsigned)chunks + (room == PANEL_ANY_ROOM ? 13u : room ? 29u : 0u)) & 63u];
  if (e.m != m || e.n_blocks != n_blocks || e.chunks != chunks || e.room != room) e = Entry{m, n_blocks, chunks, room, search_panel<Fmt>(m, n_blocks, chunks, room)};
  return e.plan;
}

// Whether an activation matrix of `rows` rows is one the panel kernel takes: it addresses the matrix with 32-bit byte
// offsets ...
inline bool panel_takes(int64_t rows, int64_t a_stride) { return rows * a_stride * 2 <= 0xffffffffll; }
// ... and writes four neighbouring output columns with one store: 8 bytes of BF16, 16 of FP32.
inline bool panel_writes(const void* out, bool f32) { return aligned(out, f32 ? 16 : 8); }

// hb_tune's cut of a dense call, where it fits (0: the estimate's): K splits and blocks of a workgroup, workgroups a tile.
struct PanelForce {
  int ks, nbw, kz;
};

// The cut of a dense call that has `room` bytes for shared tiles' partial results (0: no tile's K is shared).
template <class Fmt>
static PanelPlan cut_panel(int m, int n_blocks, int chunks, size_t room, const PanelForce& force) {
  PanelPlan q = plan_panel<Fmt>(m, n_blocks, chunks, room ? PANEL_ANY_ROOM : 0);
  if (panel_room(q) > room) q = plan_panel<Fmt>(m, n_blocks, chunks, room);
  if (force.ks || force.kz) {
    PanelPlan f = q;
    if (force.ks) {
      f.ks = force.ks;
      f.nbw = std::max(1, force.nbw);
    }
    f.groups = (n_blocks + f.nbw - 1) / f.nbw;
    f.tiles = (int64_t)f.groups * ((m + 16 * f.mt - 1) / (16 * f.mt));
    f.kz = std::max(1, std::min(force.kz, chunks / f.ks));
    f.full = f.kz > 1 ? 0 : f.tiles;
    if (f.ks * f.nbw <= PANEL_WAVES && !(f.ks & (f.ks - 1)) && f.ks <= chunks / f.kz && f.nbw >= panel_least_blocks(f.mt) && panel_lds_bytes<Fmt>(f.mt, f.ks, f.nbw) <= PANEL_LDS &&
        panel_room(f) <= room && (f.kz == 1 || f.tiles <= PANEL_SHARED_TILES))
      q = f;
  }
  return q;
}

// A dense call of p.m rows by the cut `q`; `workspace`: the room that the cut asks for (panel_room).
template <class Fmt, int EPI>
static int launch_panel(StreamParams& p, const PanelPlan& q, void* workspace, hipStream_t stream) {
  const size_t lds = panel_lds_bytes<Fmt>(q.mt, q.ks, q.nbw);
  const int64_t grid = q.full + (q.tiles - q.full) * q.kz;
  if (q.us > 1e29 || grid > 0x7fffffff) return HB_EINVAL;
  p.ks = q.ks;
  p.nbw = q.nbw;
  set_split(p);
  p.slot_rows = 16 * q.mt;
  p.a_bytes = (uint32_t)((int64_t)p.m * p.a_stride * 2);
  p.panel_groups = q.groups;
  p.panel_slots = q.slots;
  p.panel_full = (int)q.full;
  p.panel_kz = q.kz;
  p.panel_tickets = static_cast<uint32_t*>(workspace) + PLAN_HEADER;
  p.partial = reinterpret_cast<float*>(static_cast<char*>(workspace) + PANEL_TICKET_BYTES);
  auto launch = [&](auto kernel) { HB_LAUNCH(kernel, dim3((unsigned)grid), dim3(64 * q.ks * q.nbw), lds, stream, p); };
  switch (q.mt) {
    case 1: launch(panel_kernel<Fmt, EPI, 1>); break;
    case 2: launch(panel_kernel<Fmt, EPI, 2>); break;
    case 3: launch(panel_kernel<Fmt, EPI, 3>); break;
    case 4: launch(panel_kernel<Fmt, EPI, 4>); break;
    case 5: launch(panel_kernel<Fmt, EPI, 5>); break;
    case 6: launch(panel_kernel<Fmt, EPI, 6>); break;
    case 7: launch(panel_kernel<Fmt, EPI, 7>); break;
    default: launch(panel_kernel<Fmt, EPI, 8>); break;
  }
  return HB_OK;
}

// The LDS of a routed call's workgroup: the panel's, or the weight rings of its light slots.
template <class Fmt>
inline size_t panel_routed_lds(int mt, int nbw) {
  return std::max(panel_lds_bytes<Fmt>(mt, 1, nbw), Fmt::LIGHT_ROWS > 0 ? (size_t)nbw * ring_bytes<typename Fmt::Ring>() : 0);
}

// The row tiles of a routed call's slots, by its rows an expert. Higher slots expand an expert's weights for more rows at a
// time; lower ones leave registers for more workgroups on a compute unit, and with few rows a product it is their starts, ends and
// waits, not the expansion, that want something beside them. Measured at 48, 80 and 128 rows a slot, the summed experts' launches or the
// whole block in us: NVFP4, 512 experts (1024, 2688) 8 rows an expert 341, 347 and 380, 18 rows 385, 399, 422, 24 rows 412, 414, 442,
// 32 rows 475, 436, 464, 52 rows 617, 535, 526; 256 experts (768, 1536) 14 rows 116, 118, 133, 40 rows 165, 151, 160, 64 rows 207, 188, 182.
// Three-bit, 512 experts (2048, 512), even routing 14 rows 223, 234, 252, 24 rows 262, 265, 277, 40 rows 324, 313, 321, 52 rows
// 421, 351, 366; skewed 14 rows 176, 171, 174, 24 rows 232, 217, 224, 52 rows 395, 351, 343; 180 experts (1664, 384) 64 rows 158, 135, 143, 90
// rows 184, 179, 167.
// 128 and 144 rows a slot, both two workgroups a compute unit: the higher one is for the experts just past 128 rows, whose last
// rows cost a second expansion of all their weights. NVFP4, 512 experts (1024, 2688) 60 rows an expert 550 and 552, 73 rows 625 and 609, 88
// rows 713 and 698, 172 rows 1199 and 1172; 128 experts (1024, 2688) 256 rows 416 and 386, 400 rows 633 and 597, 1408 rows 1998 and
// 1928; blocks of 130 to 400 rows an expert, seventeen sizes, 0.956 to 1.022 times as long with the higher ones, 0.977 on average.
// Three-bit, 200 experts (2048, 512), even routing 75 rows 186.3 and 187.6, 90 rows 204.7 and 205.6, 130 rows 275 and 249, 150 rows 316 and
// 303, skewed 90 rows 224 and 217; 64 experts 352 rows 204 and 192, 1000 rows 495 and 480, 1408 rows 696 and 678; 96 experts (2560, 768) 512
// rows 626 and 631, 400 rows 530 and 493.
// Where slots of 128 rows all run at once (two workgroups on each of 256 compute units), higher ones only make each of them longer, but
// for the experts that one of them holds: fourteen shapes of both formats, 145 to 1000 rows an expert, 1.02 times as long with the
// higher ones on average (64 experts (1024, 256) 330 rows 85.2 and 87.5; 32 experts (2048, 512) 290 rows 110.5 and 114.4), 0.97 past one round.
// And more, lower slots start more workgroups: the three-bit format's 80 rows serve up to 60 rows an expert there (128 experts (2048,
// 512) 56 rows 99 and, of 128 rows, 102, 64 rows 115 and 102) and up to 72 elsewhere (512 experts (2048, 512), even and skewed, 68 rows 332, 346
// and 380, 396, 76 rows 379, 365; 180 experts (1664, 384) 72 rows 110, 119 and 117, 122; 256 experts (2560, 768) 72 rows 317, 319 and 350, 364).
constexpr int PANEL_SLOT_TILES = 9;      // at most
constexpr int PANEL_REFUSED_ROWS = 128;  // calls of more than MAX_SLOTS slots are refused; of higher slots, as many rows as of these
constexpr int64_t PANEL_MAX_SLOTS = 65535;
// pairs / named: the rows an expert; `experts` of the `named` are here, whose fc1 has n_blocks blocks.
template <class Fmt>
inline int panel_height(int64_t pairs, int64_t named, int experts, int shared_rows, int n_blocks) {
  constexpr int AT_ONCE = 2 * 256;  // workgroups of 128-row slots, one a slot and four blocks
  const int64_t rows = pairs * experts / named + shared_rows, slots = rows / 128 + experts / 2;  // (half a slot an expert is not full)
  const bool at_once = slots * ((n_blocks + 3) / 4) <= AT_ONCE;
  const int tiles = pairs < Fmt::LOW_ROWS * named                                            ? 3
                    : pairs < (at_once ? Fmt::MIDDLE_ROWS : Fmt::MIDDLE_ROWS_LARGE) * named  ? 5
                    : pairs < Fmt::HIGH_ROWS * named || (at_once && pairs > 144 * named)     ? 8
                                                                                             : PANEL_SLOT_TILES;
  // the ids may all lie here, whatever share of the experts this is: a call that low slots would have refused takes higher ones
  return tiles < 8 && moe_max_slots(pairs, experts, shared_rows, 16 * tiles) > PANEL_MAX_SLOTS ? 8 : tiles;
}

// What a routed call's launch needs of `p`; the workgroups of a slot. Four wavefronts a workgroup on four
// blocks, two to four workgroups a compute unit: one's start and end lie beside the others' products.
inline int panel_routed(StreamParams& p, int tiles, int64_t slots, int64_t a_rows) {
  p.ks = 1;
  p.nbw = 4;
  set_split(p);
  p.slot_rows = 16 * tiles;
  p.panel_groups = (p.n_blocks + p.nbw - 1) / p.nbw;
  p.a_bytes = (uint32_t)(a_rows * p.a_stride * 2);
  p.panel_full = (int)slots;
  return panel_takes(a_rows, p.a_stride) ? HB_OK : HB_EINVAL;
}

// Whether fc1 (`p1`) and fc2 (`p2`) of `experts` experts share a launch. One launch starts fc2's workgroups where fc1's leave room, several on one
// compute unit, and where they are few and long (once over the device at most, K of seventeen chunks and twice fc1's) and could not all stand
// there from the start, their length is the call's end; a launch of their own spreads them out. Measured, two launches and one, the routed call,
// even and (skewed) routing, us: NVFP4, 64 experts (1024, 8192), 8 rows an expert 148 and 160 (154 and 167), 28 rows 176 and 217 (220 and 246); 128 (1024, 4096) 8 rows 127
// and 132 (135 and 138); 128 (896, 2688) 5 rows 86 and 91 (85 and 86); three-bit, 64 (2048, 6144) 16 rows 273 and 296 (278 and 280), 40 rows 368 and 383 (403 and 410); 24
// (2048, 6144) 30 rows 167 and 184 (196 and 191); 32 (2048, 4096) 16 rows 112 and 118 (121 and 124), 40 rows 145 and 142 (170 and 165); NVFP4, 160 (640, 2304) 10 rows 78 and 81 (80 and 85), 60 rows 116 and 124 (146 and 134). On the other sides
// of the line: 128 (768, 2048) 10 rows 67 and 63 (72 and 70), 512 (1024, 2688) 8 rows 313 and 311 (308 and 304), 200 (896, 2048) 6 rows 101 and 96, 48 (768, 2816) 16 rows 58 and 55, three-bit 96 (2048, 2048) 7 rows 116 and 112.
inline bool panel_together(const StreamParams& p1, const StreamParams& p2, int64_t experts, int tiles) {
  const int64_t groups1 = (p1.n_blocks + 3) / 4, groups2 = (p2.n_blocks + 3) / 4;
  const bool long_end = p2.chunks >= 17 && p2.chunks >= 2 * p1.chunks && experts * groups2 <= 1024;
  return !long_end || experts * (groups1 + groups2) <= (tiles <= 3 ? 1024 : 1280);
}

// Over a plan's slots of 16 `tiles` rows; `a_rows`: rows of the activation matrix.
template <class Fmt, int EPI>
static int launch_panel_routed(StreamParams& p, int tiles, int64_t slots, int64_t a_rows, hipStream_t stream) {
  if (int e = panel_routed(p, tiles, slots, a_rows)) return e;
  const int64_t grid = (slots + 7) / 8 * 8 * p.panel_groups;
  if (grid > 0x7fffffff) return HB_EINVAL;
  auto launch = [&](auto kernel) { HB_LAUNCH(kernel, dim3((unsigned)grid), dim3(64 * p.ks * p.nbw), panel_routed_lds<Fmt>(tiles, p.nbw), stream, p); };
  tiles == 3 ? launch(panel_tile_kernel<Fmt, EPI, 3>) : tiles == 5 ? launch(panel_tile_kernel<Fmt, EPI, 5>) : tiles == 8 ? launch(panel_tile_kernel<Fmt, EPI, 8>) : launch(panel_tile_kernel<Fmt, EPI, PANEL_SLOT_TILES>);
  return HB_OK;
}

// Both layers of a call of `rows1` rows and `rows2` pairs (`plan`: the call's, whose counters the plan's launch has cleared). fc2 follows by the
// slots whose fc1 workgroups fill the device twice: started sooner they stand waiting in fc1's places (three-bit, 512 experts (2048, 512) 1543
// rows, of 85 slots a die 8 behind 247 us, 16 229, 24 217, 48 216; NVFP4, 512 (1024, 2688) 2048 rows, of 68, 4 704, 12 694 to 700, 32 702).
template <class Fmt, int EPI1>
static int launch_panel_fc12(StreamParams& p1, StreamParams& p2, int32_t* plan, int tiles, int64_t slots, int64_t rows1, int64_t rows2, int lag_forced, hipStream_t stream) {
  if (int e = panel_routed(p1, tiles, slots, rows1)) return e;
  if (int e = panel_routed(p2, tiles, slots, rows2)) return e;
  const int rounds = (int)((slots + 7) / 8), both = p1.panel_groups + p2.panel_groups;
  if ((int64_t)rounds * 8 * both > 0x7fffffff) return HB_EINVAL;
  moe_await_slots(p1, p2, plan, slots, p1.panel_groups);
  const int resident = 256 * (tiles <= 3 ? 4 : tiles <= 5 ? 3 : 2);
  const int lag = std::min(rounds, lag_forced ? lag_forced : std::max(1, 2 * resident / (8 * p1.panel_groups)));
  auto launch = [&](auto kernel) {
    HB_LAUNCH(kernel, dim3((unsigned)(8 * rounds * both)), dim3(64 * p1.nbw), panel_routed_lds<Fmt>(tiles, p1.nbw), stream, p1, p2, rounds, lag);
  };
  tiles == 3 ? launch(panel_fc12_tile_kernel<Fmt, EPI1, 3>) : tiles == 5 ? launch(panel_fc12_tile_kernel<Fmt, EPI1, 5>) : tiles == 8 ? launch(panel_fc12_tile_kernel<Fmt, EPI1, 8>) : launch(panel_fc12_tile_kernel<Fmt, EPI1, PANEL_SLOT_TILES>);
  return HB_OK;
}

}  // namespace hb
