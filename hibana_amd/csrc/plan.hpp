// The expert plan of a routed call (device code shared by the plan's own launches and by kernels that plan beside other work).
#pragma once

#include "route.hpp"
#include "stream_common.hpp"

namespace hb {

// ---------------------------------------------------------------------------------------------------- expert plan
//
// The expert-sorted pair list of a routed call (the reference's prep kernel, hibana/kernels/csrc/w3_gemm.cu:710-782):
// distinct local experts in ascending id, each expert's pairs in ascending pair index (a stable sort), cut into slots
// of at most 16 rows. One workgroup; any number of pairs. Integer atomics on LDS counters only (order-independent).
//   plan[0] = slots, plan[1] = distinct experts, plan[2] = kept routed pairs,
//   plan[16 + 4 s ..] = { local expert id (-1: the shared expert), first sorted position, rows, 0 }: the shared
//                        expert's slots first, then the routed experts' (the heavily loaded ones before the others)
//   order[pos] = pair index (row * topk + slot; shared expert rows: pairs + row)
constexpr int PLAN_THREADS = 1024;
constexpr int PLAN_WAVES = PLAN_THREADS / 64;
constexpr int PLAN_BATCH = 8;  // tiles of 64 pairs whose ids a wavefront requests at once
constexpr int PLAN_WIDE_PAIRS = 8192;   // from this many pairs they are counted by several workgroups in a launch of its own
constexpr int PLAN_WIDE_GROUPS = 64;
// Up to this many rows the plan's workgroup routes them itself (one a wavefront): no ticket, no second workgroup to wait for, but the
// rows share one compute unit. The three-bit layer, rows of 10 of 512 experts, even and skewed routing, us, routed there and in workgroups
// of their own (moe_route_plan_kernel): two rows 28.4, 27.6 and 28.7, 28.0; three 29.1, 28.5 and 29.9, 28.8; four 31.6, 29.1 and 32.1, 29.6;
// five 34.3, 32.8 and 34.2, 32.8; the latent block, 22 of 512, two rows 63.1 and 63.8, four 81.6 and 82.6, five 91.8 and 91.0.
constexpr int ROUTE_FUSED_ROWS = 4;
// Up to this many pairs of such rows one wavefront plans, above them plan_by_rows: its steps go by the pairs. In the same order, one
// wavefront and by rows: two rows of ten 28.4 and 28.1, 27.8 and 27.7, of 22 65.8 and 63.1; three of ten 30.4 and 29.1, 29.2 and 28.4; four 33.8
// and 31.6, 30.4 and 29.1; of eight of 256 experts two 26.5 and 26.7, three 27.5 and 27.3.
constexpr int ROUTE_FEW_PAIRS = 24;

struct Scan3 {
  int a, b, c;
};

// Exclusive scan over the workgroup of two words a thread whose four 16-bit halves are sums of their own (none reaches
// 65536, so no carry crosses a half): one DPP scan a word in each wavefront, the wavefronts' totals through LDS, one
// barrier. `total` receives the two sums. scratch: 2 * PLAN_WAVES ints, not in use by anyone before the call's barrier.
struct Scan2 {
  int lo, hi;
};
__device__ __forceinline__ Scan2 block_exclusive_scan2(Scan2 v, int* scratch, Scan2* total) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, waves = blockDim.x >> 6;
  const int lo = wave_inclusive_sum(v.lo), hi = wave_inclusive_sum(v.hi);
  if (lane == 63) {
    scratch[wave] = lo;
    scratch[PLAN_WAVES + wave] = hi;
  }
  __syncthreads();
  int before_lo = 0, before_hi = 0, all_lo = 0, all_hi = 0;
  for (int w = 0; w < waves; w++) {  // the same address in every lane: broadcast reads
    const int a = scratch[w], b = scratch[PLAN_WAVES + w];
    before_lo += w < wave ? a : 0;
    before_hi += w < wave ? b : 0;
    all_lo += a;
    all_hi += b;
  }
  total->lo = all_lo;
  total->hi = all_hi;
  return Scan2{before_lo + lo - v.lo, before_hi + hi - v.hi};
}

// Exclusive scan of three integers per thread over the workgroup at once; `total` receives the three sums.
__device__ __forceinline__ Scan3 block_exclusive_scan3(Scan3 v, int* scratch /* 3 * (PLAN_WAVES + 1) ints */, Scan3* total) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const Scan3 inc{wave_inclusive_sum(v.a), wave_inclusive_sum(v.b), wave_inclusive_sum(v.c)};
  __syncthreads();  // scratch may still be read from a previous scan
  if (lane == 63) {
    scratch[wave] = inc.a;
    scratch[PLAN_WAVES + wave] = inc.b;
    scratch[2 * PLAN_WAVES + wave] = inc.c;
  }
  __syncthreads();
  Scan3 before{0, 0, 0}, all{0, 0, 0};
#pragma unroll
  for (int w = 0; w < PLAN_WAVES; w++) {  // the same address in every lane: broadcast reads
    const int a = scratch[w], b = scratch[PLAN_WAVES + w], c = scratch[2 * PLAN_WAVES + w];
    before.a += w < wave ? a : 0;
    before.b += w < wave ? b : 0;
    before.c += w < wave ? c : 0;
    all.a += a;
    all.b += b;
    all.c += c;
  }
  *total = all;
  return Scan3{before.a + inc.a - v.a, before.b + inc.b - v.b, before.c + inc.c - v.c};
}

// The plan of at most 64 pairs (a decode step), by one wavefront, a pair a lane: no counters per expert, no scan over
// the experts. Lanes with the same expert find each other by ballots over the id's bits; what precedes an expert in
// either order (sorted positions: ascending id; slot table: shared, heavily loaded, the rest) is summed in a loop over
// the lanes. Writes exactly what the general form writes.
__device__ __forceinline__ void plan_few_pairs(const int32_t* ids, int pairs, int e_lo, int e_n, int shared_rows, int32_t* __restrict__ plan,
                                               int32_t* __restrict__ order, int slot_rows, int slot_cap) {
  const int lane = threadIdx.x & 63;
  int e = lane < pairs ? load_through(&ids[lane]) - e_lo : -1;
  if (e < 0 || e >= e_n) e = -1;
  int id_bits = 1;
  while ((1 << id_bits) < e_n) id_bits++;
  uint64_t same = __ballot(e >= 0);
  const int kept = __popcll(same);
  for (int b = 0; b < id_bits; b++) {
    const uint64_t m = __ballot((e >> b) & 1);
    same &= ((e >> b) & 1) ? m : ~m;
  }
  const int rank = __popcll(same & ((1ull << lane) - 1ull)), count = e >= 0 ? __popcll(same) : 0;
  const bool first = e >= 0 && rank == 0;
  const int my_slots = (count + slot_rows - 1) / slot_rows;
  const bool heavy = 4 * count > slot_rows;
  int start = 0, heavy_before = 0, light_before = 0, heavy_total = 0, light_total = 0, distinct = 0;
  for (int j = 0; j < pairs; j++) {  // uniform: lane j's expert, if lane j is the first of it
    const int ej = __builtin_amdgcn_readlane(first ? e : -1, j);
    if (ej < 0) continue;
    const int cj = __builtin_amdgcn_readlane(count, j), sj = __builtin_amdgcn_readlane(my_slots, j);
    const bool hj = 4 * cj > slot_rows;
    distinct++;
    heavy_total += hj ? sj : 0;
    light_total += hj ? 0 : sj;
    if (ej < e) {
      start += cj;
      heavy_before += hj ? sj : 0;
      light_before += hj ? 0 : sj;
    }
  }
  const int shared_slots = (shared_rows + slot_rows - 1) / slot_rows;
  const int slots = shared_slots + heavy_total + light_total;
  if (e >= 0) order[start + rank] = lane;
  if (first) {
    const int my_slot = shared_slots + (heavy ? heavy_before : heavy_total + light_before);
    for (int s = 0; s < my_slots; s++) {
      int32_t* entry = plan + PLAN_HEADER + 4 * (my_slot + s);
      entry[0] = e;
      entry[1] = start + s * slot_rows;
      entry[2] = min(slot_rows, count - s * slot_rows);
      entry[3] = 0;
    }
  }
  for (int s = lane; s < shared_slots; s += 64) {
    int32_t* entry = plan + PLAN_HEADER + 4 * s;
    entry[0] = -1;
    entry[1] = kept + s * slot_rows;
    entry[2] = min(slot_rows, shared_rows - s * slot_rows);
    entry[3] = 0;
  }
  for (int r = lane; r < shared_rows; r += 64) order[kept + r] = pairs + r;
  for (int s = slots + lane; s < slot_cap; s += 64) {
    int32_t* entry = plan + PLAN_HEADER + 4 * s;
    entry[0] = entry[1] = entry[2] = entry[3] = 0;
  }
  for (int s = lane; s < slot_cap; s += 64) plan_done(plan, slot_cap)[s * DONE_PITCH] = 0;
  if (lane == 0) {
    plan[0] = slots;
    plan[1] = distinct;
    plan[2] = kept;
  }
}

// What every form of the plan writes behind the experts' slots: the shared expert's slots and rows, "no rows" in the
// entries the launches' grids reach beyond the last slot (a workgroup learns that it has nothing to do from its own
// entry, without a second dependent read of the count), the slots' arrival counters at zero, the header.
__device__ __forceinline__ void plan_tail(int32_t* __restrict__ plan, int32_t* __restrict__ order, int pairs, int shared_rows, int slot_rows, int slot_cap,
                                          int slots, int distinct, int kept, bool counters = true) {
  const int shared_slots = (shared_rows + slot_rows - 1) / slot_rows;
  for (int s = threadIdx.x; s < shared_slots; s += blockDim.x) {
    int32_t* entry = plan + PLAN_HEADER + 4 * s;
    entry[0] = -1;
    entry[1] = kept + s * slot_rows;
    entry[2] = min(slot_rows, shared_rows - s * slot_rows);
    entry[3] = 0;
  }
  for (int r = threadIdx.x; r < shared_rows; r += blockDim.x) order[kept + r] = pairs + r;
  for (int s = slots + threadIdx.x; s < slot_cap; s += blockDim.x) {
    int32_t* entry = plan + PLAN_HEADER + 4 * s;
    entry[0] = entry[1] = entry[2] = entry[3] = 0;
  }
  if (counters)
    for (int s = threadIdx.x; s < slot_cap; s += blockDim.x) plan_done(plan, slot_cap)[s * DONE_PITCH] = 0;
  if (threadIdx.x == 0) {
    plan[0] = slots;
    plan[1] = distinct;
    plan[2] = kept;
  }
}

// The plan of a call of at most PLAN_ROWS_MAX rows in which no row names an expert twice (the library's own routing
// of a decode or verify call), by one workgroup of PLAN_THREADS: an expert's rows are one bit each of a 64-bit word in
// LDS (integer ORs: their order does not matter), its pair count is the word's population, and a pair's place among
// its expert's is the population below its row's bit - ascending pair index, as the general form places them. One
// trip to memory for the ids (every thread's loads asked for together), one scan, no per-tile matching. Writes
// exactly what plan_work writes.
constexpr int PLAN_ROWS_MAX = 64;
constexpr int PLAN_ROWS_PER_THREAD = 4;  // 64 rows of at most 64 selections over 1024 threads
__device__ __forceinline__ void plan_by_rows(const int32_t* ids, int rows, int topk, int e_lo, int e_n, int shared_rows, int32_t* __restrict__ plan,
                                             int32_t* __restrict__ order, int slot_rows, int slot_cap, int* lds, bool cleared = false) {
  uint32_t* occ_lo = reinterpret_cast<uint32_t*>(lds);  // [e_n] rows 0 .. 31 that name expert e
  uint32_t* occ_hi = occ_lo + e_n;                      // [e_n] rows 32 .. 63
  int* start = lds + 2 * e_n;                           // [e_n] first sorted position of expert e
  int* scratch = start + e_n;                           // [2 * PLAN_WAVES]
  const int pairs = rows * topk;
  int mine[PLAN_ROWS_PER_THREAD], row_of[PLAN_ROWS_PER_THREAD];
#pragma unroll
  for (int j = 0; j < PLAN_ROWS_PER_THREAD; j++) {  // asked for before anything else is done
    const int q = threadIdx.x + j * PLAN_THREADS;
    mine[j] = q < pairs ? load_through(&ids[q]) - e_lo : -1;
  }
  for (int e = threadIdx.x; e < 2 * e_n; e += PLAN_THREADS) occ_lo[e] = 0u;
#pragma unroll
  for (int j = 0; j < PLAN_ROWS_PER_THREAD; j++) row_of[j] = (threadIdx.x + j * PLAN_THREADS) / topk;
  __syncthreads();
#pragma unroll
  for (int j = 0; j < PLAN_ROWS_PER_THREAD; j++) {
    if (mine[j] < 0 || mine[j] >= e_n) mine[j] = -1;
    if (mine[j] >= 0) atomicOr(row_of[j] < 32 ? &occ_lo[mine[j]] : &occ_hi[mine[j]], 1u << (row_of[j] & 31));
  }
  __syncthreads();
  const int e = threadIdx.x;  // one thread an expert: the launch keeps e_n <= PLAN_THREADS
  const int count = e < e_n ? __popc(occ_lo[e]) + __popc(occ_hi[e]) : 0;  // at most 64
  const int my_slots = (count + slot_rows - 1) / slot_rows;
  const bool heavy = 4 * count > slot_rows;
  // four sums in two words: rows (at most 4096) and light slots; heavy slots and distinct experts (at most 1024 each)
  Scan2 tot;
  const Scan2 at = block_exclusive_scan2(Scan2{count | (heavy ? 0 : my_slots) << 16, (heavy ? my_slots : 0) | (count > 0 ? 1 << 16 : 0)}, scratch, &tot);
  const int shared_slots = (shared_rows + slot_rows - 1) / slot_rows;
  const int kept = tot.lo & 0xffff, distinct = tot.hi >> 16, heavy_slots = tot.hi & 0xffff;
  const int slots = shared_slots + heavy_slots + (tot.lo >> 16);
  if (e < e_n) {
    const int my_start = at.lo & 0xffff;
    start[e] = my_start;
    const int my_slot = shared_slots + (heavy ? (at.hi & 0xffff) : heavy_slots + (at.lo >> 16));
    for (int s = 0; s < my_slots; s++) {
      int32_t* entry = plan + PLAN_HEADER + 4 * (my_slot + s);
      entry[0] = e;
      entry[1] = my_start + s * slot_rows;
      entry[2] = min(slot_rows, count - s * slot_rows);
      entry[3] = 0;
    }
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < PLAN_ROWS_PER_THREAD; j++) {
    if (mine[j] < 0) continue;
    const int r = row_of[j];
    const uint32_t lo = occ_lo[mine[j]], hi = occ_hi[mine[j]];
    const int below = r < 32 ? __popc(lo & ((1u << r) - 1u)) : __popc(lo) + __popc(hi & ((1u << (r - 32)) - 1u));
    order[start[mine[j]] + below] = threadIdx.x + j * PLAN_THREADS;
  }
  // `cleared`: the launch's other workgroups have already put "no rows" into every entry and zeroed the arrival counters
  plan_tail(plan, order, pairs, shared_rows, slot_rows, cleared ? slots : slot_cap, slots, distinct, kept, !cleared);
}

// The plan itself, by one workgroup of PLAN_THREADS (`group` of `groups` when many pairs are shared): `lds` is the
// launch's dynamic LDS.
template <bool WIDE>  // false: one workgroup (phase 0) and nothing of the shared form compiled in
__device__ __forceinline__ void plan_work(const int32_t* ids, int pairs, int e_lo, int e_n, int shared_rows, int32_t* __restrict__ plan,
                                          int32_t* __restrict__ order, int slot_rows, int slot_cap, int32_t* __restrict__ wide, int groups_, int phase_,
                                          int group_, int* lds) {
  const int groups = WIDE ? groups_ : 1, phase = WIDE ? phase_ : 0;
  if (!WIDE && pairs <= 64) {  // a decode step: one wavefront plans it
    if (threadIdx.x < 64) plan_few_pairs(ids, pairs, e_lo, e_n, shared_rows, plan, order, slot_rows, slot_cap);
    return;
  }
  int* seg_count = lds;                         // [PLAN_WAVES][e_n]: pairs of expert e in segment w, then running positions
  int* start = lds + PLAN_WAVES * e_n;          // [e_n]: first sorted position of expert e
  int* scratch = start + e_n;                   // [3 * (PLAN_WAVES + 1)]
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, group = WIDE ? group_ : 0;
  // segment (group, w) = pairs [(group * PLAN_WAVES + w) * seg, ... + seg), seg a multiple of 64
  const int seg = (((pairs + groups - 1) / groups + PLAN_WAVES - 1) / PLAN_WAVES + 63) / 64 * 64;
  const int lo = min(pairs, (group * PLAN_WAVES + wave) * seg), hi = min(pairs, lo + seg);
  const int batch = seg > 64 ? PLAN_BATCH : 1;  // long segments: the ids of a batch of tiles are requested together
  const int nseg = WIDE ? PLAN_WAVES : min(PLAN_WAVES, (pairs + seg - 1) / seg);  // segments that hold pairs: the others' counters are neither cleared nor read
  const int e = threadIdx.x;  // one thread an expert: the launch keeps e_n <= PLAN_THREADS
  if (phase != 2) {
    for (int i = threadIdx.x; i < nseg * e_n; i += PLAN_THREADS) seg_count[i] = 0;
    __syncthreads();
  }
  int only = -1;  // seg == 64: the local expert of this lane's one pair, kept for the placement (no second read of the ids)
  for (int i0 = lo + lane; phase != 2 && i0 < hi; i0 += 64 * batch) {
    if (batch == 1) {
      const int e = load_through(&ids[i0]) - e_lo;
      if (e >= 0 && e < e_n) {
        atomicAdd(&seg_count[wave * e_n + e], 1);
        only = e;
      }
      continue;
    }
    int e[PLAN_BATCH];
#pragma unroll
    for (int j = 0; j < PLAN_BATCH; j++) e[j] = i0 + 64 * j < hi ? load_through(&ids[i0 + 64 * j]) - e_lo : -1;
#pragma unroll
    for (int j = 0; j < PLAN_BATCH; j++)
      if (e[j] >= 0 && e[j] < e_n) atomicAdd(&seg_count[wave * e_n + e[j]], 1);
  }
  __syncthreads();
  if (phase == 1) {  // this group's pairs of each expert
    if (e < e_n) {
      int count = 0;
      for (int wv = 0; wv < PLAN_WAVES; wv++) count += seg_count[wv * e_n + e];
      wide[group * e_n + e] = count;
    }
    return;
  }
  if (phase == 3) {  // the first position of each of this group's segments' runs, from the group's own
    if (e < e_n) {
      int run = wide[group * e_n + e];
      for (int wv = 0; wv < PLAN_WAVES; wv++) {
        const int c = seg_count[wv * e_n + e];
        seg_count[wv * e_n + e] = run;
        run += c;
      }
    }
    __syncthreads();
  } else {
  // Slot order is the order the hardware starts a launch's workgroups in, so the long-running slots go first: the
  // shared expert's (full slots), then the experts with more than a quarter slot of rows, then the rest, each class in
  // ascending expert id. Sorted positions are another matter: ascending expert id, the shared rows after the routed
  // pairs.
  const int shared_slots = (shared_rows + slot_rows - 1) / slot_rows;
  int count = 0;
  int of_group[PLAN_WIDE_GROUPS];  // phase 2: the groups' counts of this thread's expert, all asked for at once
  if (e < e_n) {
    if (phase == 0) {
      for (int wv = 0; wv < nseg; wv++) count += seg_count[wv * e_n + e];
    } else {
#pragma unroll
      for (int g = 0; g < PLAN_WIDE_GROUPS; g++) of_group[g] = g < groups ? wide[g * e_n + e] : 0;
#pragma unroll
      for (int g = 0; g < PLAN_WIDE_GROUPS; g++) count += of_group[g];
    }
  }
  const int my_slots = (count + slot_rows - 1) / slot_rows;
  const bool heavy = 4 * count > slot_rows;
  Scan3 tot;  // a: rows; b: heavy slots, and distinct experts in the upper half (neither sum reaches 65536); c: light slots
  const Scan3 at = block_exclusive_scan3(Scan3{count, (heavy ? my_slots : 0) | (count > 0 ? 1 << 16 : 0), heavy ? 0 : my_slots}, scratch, &tot);
  const int kept = tot.a, distinct = tot.b >> 16, heavy_slots = tot.b & 0xffff;
  const int slots = shared_slots + heavy_slots + tot.c;
  if (e < e_n) {
    const int my_start = at.a, my_slot = shared_slots + (heavy ? (at.b & 0xffff) : heavy_slots + at.c);
    start[e] = my_start;
    for (int s = 0; s < my_slots; s++) {
      int32_t* entry = plan + PLAN_HEADER + 4 * (my_slot + s);
      entry[0] = e;
      entry[1] = my_start + s * slot_rows;
      entry[2] = min(slot_rows, count - s * slot_rows);
      entry[3] = 0;
    }
    // turn the per-segment (phase 2: per-group) counts into the first position of each segment's (group's) run
    int run = my_start;
    if (phase == 0) {
      for (int wv = 0; wv < nseg; wv++) {
        const int c = seg_count[wv * e_n + e];
        seg_count[wv * e_n + e] = run;
        run += c;
      }
    } else {
#pragma unroll
      for (int g = 0; g < PLAN_WIDE_GROUPS; g++) {
        if (g < groups) wide[g * e_n + e] = run;
        run += of_group[g];
      }
    }
  }
  __syncthreads();
  plan_tail(plan, order, pairs, shared_rows, slot_rows, slot_cap, slots, distinct, kept);
  if (phase == 2) return;
  }
  // stable placement: each wavefront walks its segment 64 pairs at a time; a lane's position is its expert's running
  // position in this segment plus the number of lower lanes of the tile with the same expert
  int id_bits = 1;
  while ((1 << id_bits) < e_n) id_bits++;
  for (int i0 = lo; i0 < hi; i0 += 64 * batch) {
    int eb[PLAN_BATCH];
#pragma unroll
    for (int j = 0; j < PLAN_BATCH; j++) {
      const int i = i0 + 64 * j + lane;
      int e;
      if (seg == 64) {  // uniform: one tile a wavefront, read when it was counted
        e = j == 0 ? only : -1;
      } else {
        e = j < batch && i < hi ? load_through(&ids[i]) - e_lo : -1;
        if (e < 0 || e >= e_n) e = -1;
      }
      eb[j] = e;
    }
#pragma unroll
    for (int j = 0; j < PLAN_BATCH; j++) {
      if (j < batch && i0 + 64 * j < hi) {  // wave-uniform: some pair of the segment is in this tile
        const int i = i0 + 64 * j + lane, e = eb[j];
        uint64_t same = __ballot(e >= 0);
        for (int b = 0; b < id_bits; b++) {
          const uint64_t m = __ballot((e >> b) & 1);
          same &= ((e >> b) & 1) ? m : ~m;
        }
        if (e >= 0) {
          const uint64_t below = same & ((1ull << lane) - 1ull);
          const int base = seg_count[wave * e_n + e];
          order[base + __popcll(below)] = i;
          const bool last = (same >> lane) == 1ull;  // the highest lane of this expert in the tile advances the counter
          if (last) seg_count[wave * e_n + e] = base + __popcll(same);
        }
      }
    }
    // the read of `base` above and the update by `last` are in the same wavefront; LDS operations of one wavefront
    // execute in program order, and the next tile's reads come after this write
  }
}

// For launches whose last workgroup plans. "No rows" into every entry of the slot table and the slots' arrival counters at
// zero, word `first` and every `step`-th after it - with stores that go through to memory and are waited for, so the words
// are there, and in no L2 as modified lines, before anyone's ticket: the planner's own stores to the entries it fills come
// after its ticket and are the only modified copies.
__device__ __forceinline__ void clear_plan(int32_t* plan, int slot_cap, int first, int step) {
  int32_t* done = plan_done(plan, slot_cap);
  for (int i = first; i < 5 * slot_cap; i += step) store_through(i < 4 * slot_cap ? plan + PLAN_HEADER + i : done + (i - 4 * slot_cap) * DONE_PITCH, 0);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}
// One thread a workgroup draws a ticket: whether it is the last of `groups`, which puts the counter back for the next call.
__device__ __forceinline__ int last_to_arrive(int32_t* plan, int groups) {
  const bool last = atomicAdd(reinterpret_cast<unsigned*>(plan + PLAN_TICKET), 1u) == (unsigned)groups - 1u;
  if (last) store_through(plan + PLAN_TICKET, 0);  // every other workgroup of this launch has drawn
  return last;
}

// What a launch that routes and plans a small latent block's rows beside other work needs to know (nvfp4.hip); false: the routing and the plan
// take launches of their own.
struct LatentPlan {
  RouteParams route;
  int groups, by_rows, slot_cap;  // workgroups that route; whether no row names an expert twice (plan_by_rows); the slot table's entries
  size_t lds;
};
bool latent_plan_of(const LatentRouter& r, LatentPlan& q);

}  // namespace hb
