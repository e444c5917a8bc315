// Kernels and host helpers shared by every routed-expert call: the expert plan, the combine, softmax top-k routing.
#include <string.h>

#include <atomic>
#include <mutex>
#include <vector>

#include "plan.hpp"
#include "route.hpp"
#include "route_budget.hpp"
#include "stream_common.hpp"

namespace hb {

// ---------------------------------------------------------------------------------------------------- routing
// (route.hpp: a row a wavefront)
template <bool SIGMOID, int PER>
__global__ __launch_bounds__(64) void route_topk_kernel(RouteParams p) {
  route_row<SIGMOID, PER>(p, blockIdx.x, threadIdx.x);
}

template <bool SIGMOID>
static void launch_route(const RouteParams& p, int m, hipStream_t stream) {
  if (p.per <= 8) {
    HB_LAUNCH((route_topk_kernel<SIGMOID, 8>), dim3((unsigned)m), dim3(64), 0, stream, p);
  } else {
    HB_LAUNCH((route_topk_kernel<SIGMOID, 16>), dim3((unsigned)m), dim3(64), 0, stream, p);
  }
}

// ---------------------------------------------------------------------------------------------------- expert plan
// (plan.hpp: by one workgroup, or a share of it)
// With `route.logits` set the workgroup first routes the route_rows rows itself (a row a wavefront: at most
// ROUTE_FUSED_ROWS) into route.ids / route.weights, which `ids` then names; `by_rows`: none of them names an expert twice.
//
// With `job.lanes` set the launch has further workgroups, which round the job's activations to E4M3 and plan nothing.
//
// Many pairs (a prefill chunk) are counted by `groups` workgroups into `wide` [groups, e_n] (phase 1), and moe_place_kernel does the rest.
// Very many (more shares than PLAN_WIDE_GROUPS), or many with a rounding job, take three launches of this kernel, `wide` between them:
// phase 1, each group counts its share of the pairs per expert; phase 2, one workgroup adds the groups' counts, writes the slot table and
// turns `wide` into the first sorted position of each group's run of each expert; phase 3, each group places its share. Phase 0 is all of
// it in one workgroup.
template <bool WIDE>
__global__ __launch_bounds__(PLAN_THREADS) void moe_plan_kernel(const int32_t* ids, int pairs, int e_lo, int e_n, int shared_rows,
                                                                int32_t* __restrict__ plan, int32_t* __restrict__ order, RouteParams route,
                                                                int route_rows, int by_rows, int slot_rows, int slot_cap, int32_t* __restrict__ wide,
                                                                int groups, int phase, QuantJob job) {
  extern __shared__ int lds[];
  if (!WIDE && blockIdx.x > 0) {  // the workgroups beside the plan's: the activation rounding
    quant_job_share(job, blockIdx.x - 1, reinterpret_cast<float*>(lds));
    return;
  }
  if (!WIDE && route.logits) {
    // (a loop over the rows keeps what no row changes in registers, and spills: latent block of four rows 83.8 us, without 82.0)
    const int r = threadIdx.x >> 6;
    if (r < route_rows) route_any(route, r, threadIdx.x & 63);
    __syncthreads();
  }
  if (!WIDE && by_rows) {
    plan_by_rows(ids, route_rows, route.k, e_lo, e_n, shared_rows, plan, order, slot_rows, slot_cap, lds);
    return;
  }
  plan_work<WIDE>(ids, pairs, e_lo, e_n, shared_rows, plan, order, slot_rows, slot_cap, wide, groups, phase, blockIdx.x, lds);
}

// The plan of more pairs than one workgroup places quickly, by workgroups that each place a share of `share` pairs (a multiple
// of 64, one pair a thread) and share nothing: every one of them learns all experts' counts, and how many of those are
// ahead of its share, for itself. Writes exactly what plan_work writes. TABLE: from the counts of the shares `wide`
// [gridDim.x, e_n] that a launch ahead of it has made (moe_plan_kernel, phase 1); else from all ids, read by each workgroup.
// What bounds it is latency: one trip to memory for the ids or counts, a histogram in LDS, the scan over the experts, the
// stores. One workgroup that plans behind the routing in its launch took 15.0 us for both at 128 rows of ten, 21.8 at 512 (a
// routing launch and this one 5.4 + 5.9 and 6.2 + 7.2); alone 14.4 us at 5632 pairs; count, scan and place as three launches 19.2 us at
// 15430 pairs, 19.8 at 45056 (count and this 12.2 and 14.7).
constexpr int PLACE_SHARE = 256, PLACE_TABLE_SHARE = PLAN_THREADS;
// Of at most PLACE_TABLE_SHARE pairs a counting workgroup, plan_work's segments are 64 pairs a wavefront: what it counts is that share.
static_assert(PLACE_TABLE_SHARE == 64 * PLAN_WAVES, "the counting workgroups' shares are the placing ones'");
template <bool TABLE>
__global__ __launch_bounds__(PLAN_THREADS) void moe_place_kernel(const int32_t* __restrict__ ids, int pairs, int e_lo, int e_n, int shared_rows,
                                                                 int32_t* __restrict__ plan, int32_t* __restrict__ order, int slot_rows, int slot_cap,
                                                                 const int32_t* __restrict__ wide) {
  constexpr int SHARE = TABLE ? PLACE_TABLE_SHARE : PLACE_SHARE, TILES = SHARE / 64;
  extern __shared__ int lds[];
  int* run = lds;                                      // [TILES][e_n]: pairs of expert e in tile w of the share, then the tile's first position
  int* total = run + TILES * e_n;                      // [e_n] (from all ids) pairs of expert e ...
  int* ahead = total + e_n;                            // [e_n] ... and those ahead of the share
  int* scratch = TABLE ? total : ahead + e_n;          // [3 * (PLAN_WAVES + 1)]
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, group = blockIdx.x, groups = gridDim.x, lo = group * SHARE;
  auto local = [&](int i) {
    const int e = i < pairs ? ids[i] - e_lo : -1;
    return e >= 0 && e < e_n ? e : -1;
  };
  const int mine = threadIdx.x < SHARE ? local(lo + threadIdx.x) : -1;
  const int e = threadIdx.x;  // one thread an expert: the launch keeps e_n <= PLAN_THREADS
  int count = 0, before = 0;
  if (TABLE) {
    constexpr int BATCH = 16;  // asked for together, without a condition
    for (int g0 = 0; g0 < groups; g0 += BATCH) {
      int of_group[BATCH];
#pragma unroll
      for (int j = 0; j < BATCH; j++) of_group[j] = wide[min(g0 + j, groups - 1) * e_n + min(e, e_n - 1)];
#pragma unroll
      for (int j = 0; j < BATCH; j++) {
        count += g0 + j < groups ? of_group[j] : 0;
        before += g0 + j < group ? of_group[j] : 0;
      }
    }
    if (e >= e_n) count = 0;
  }
  for (int i = threadIdx.x; i < (TABLE ? TILES : TILES + 2) * e_n; i += PLAN_THREADS) lds[i] = 0;
  __syncthreads();
  if (!TABLE) {
    for (int i0 = threadIdx.x; i0 < pairs; i0 += PLAN_THREADS * PLAN_BATCH) {
      int of[PLAN_BATCH];
#pragma unroll
      for (int j = 0; j < PLAN_BATCH; j++) of[j] = local(i0 + j * PLAN_THREADS);
#pragma unroll
      for (int j = 0; j < PLAN_BATCH; j++)
        if (of[j] >= 0) {
          atomicAdd(&total[of[j]], 1);
          if (i0 + j * PLAN_THREADS < lo) atomicAdd(&ahead[of[j]], 1);
        }
    }
  }
  // the lanes of a tile that name the same expert, by ballots over the id's bits
  int rank = 0;
  if (wave < TILES) {
    int id_bits = 1;
    while ((1 << id_bits) < e_n) id_bits++;
    uint64_t same = __ballot(mine >= 0);
    for (int b = 0; b < id_bits; b++) {
      const uint64_t m = __ballot((mine >> b) & 1);
      same &= ((mine >> b) & 1) ? m : ~m;
    }
    rank = __popcll(same & ((1ull << lane) - 1ull));
    if (mine >= 0 && rank == 0) run[wave * e_n + mine] = __popcll(same);
  }
  __syncthreads();
  if (!TABLE && e < e_n) count = total[e], before = ahead[e];
  const int my_slots = (count + slot_rows - 1) / slot_rows, shared_slots = (shared_rows + slot_rows - 1) / slot_rows;
  const bool heavy = 4 * count > slot_rows;
  Scan3 tot;  // as in plan_work
  const Scan3 at = block_exclusive_scan3(Scan3{count, (heavy ? my_slots : 0) | (count > 0 ? 1 << 16 : 0), heavy ? 0 : my_slots}, scratch, &tot);
  const int kept = tot.a, heavy_slots = tot.b & 0xffff, slots = shared_slots + heavy_slots + tot.c;
  if (e < e_n) {
    int first = at.a + before;
#pragma unroll
    for (int w = 0; w < TILES; w++) {
      const int c = run[w * e_n + e];
      run[w * e_n + e] = first;
      first += c;
    }
  }
  __syncthreads();
  if (mine >= 0) order[run[wave * e_n + mine] + rank] = lo + threadIdx.x;
  // what is written once, dealt out to the workgroups
  if (e < e_n && e % groups == group) {
    const int my_slot = shared_slots + (heavy ? (at.b & 0xffff) : heavy_slots + at.c);
    for (int s = 0; s < my_slots; s++) {
      int32_t* entry = plan + PLAN_HEADER + 4 * (my_slot + s);
      entry[0] = e;
      entry[1] = at.a + s * slot_rows;
      entry[2] = min(slot_rows, count - s * slot_rows);
      entry[3] = 0;
    }
  }
  const int first = group * PLAN_THREADS + threadIdx.x, step = groups * PLAN_THREADS;
  for (int s = first; s < shared_slots; s += step) {
    int32_t* entry = plan + PLAN_HEADER + 4 * s;
    entry[0] = -1;
    entry[1] = kept + s * slot_rows;
    entry[2] = min(slot_rows, shared_rows - s * slot_rows);
    entry[3] = 0;
  }
  for (int r = first; r < shared_rows; r += step) order[kept + r] = pairs + r;
  for (int s = slots + first; s < slot_cap; s += step) {
    int32_t* entry = plan + PLAN_HEADER + 4 * s;
    entry[0] = entry[1] = entry[2] = entry[3] = 0;
  }
  for (int s = first; s < slot_cap; s += step) plan_done(plan, slot_cap)[s * DONE_PITCH] = 0;
  if (first == 0) {
    plan[0] = slots;
    plan[1] = tot.b >> 16;
    plan[2] = kept;
  }
}

// Routing and plan of a verify-sized call in ONE launch: `route_groups` workgroups route `group_rows` rows each (a
// row a wavefront, spread over the device, as the routing launch does), and the one that finishes last plans - it
// learns that it is the last from an arrival counter in the call's own workspace (plan[PLAN_TICKET]: zero when the
// caller hands the workspace over, put back to zero by every last arriver, as the split-K counters of the reference's
// dense kernel are, hibana/kernels/csrc/w3_gemm.cu:230-240), so calls in flight together, each on a workspace of its
// own, share nothing. A workgroup's ids are written through to memory and waited for before its ticket is drawn, and
// the plan reads ids past its own L2 (store_through / load_through): no cache write-back, no invalidate. Nobody
// waits: a workgroup that is not the last leaves. `by_rows`: the rows name no expert twice and are at most
// PLAN_ROWS_MAX (plan_by_rows). Workgroups past the routing ones round the job's activations, as in moe_plan_kernel.
__global__ __launch_bounds__(PLAN_THREADS) void moe_route_plan_kernel(const int32_t* ids, int pairs, int e_lo, int e_n, int shared_rows,
                                                                      int32_t* __restrict__ plan, int32_t* __restrict__ order, RouteParams route,
                                                                      int route_rows, int route_groups, int group_rows, int by_rows, int slot_rows,
                                                                      int slot_cap, QuantJob job) {
  extern __shared__ int lds[];
  __shared__ int last;
  if ((int)blockIdx.x >= route_groups) {
    quant_job_share(job, blockIdx.x - route_groups, reinterpret_cast<float*>(lds));
    return;
  }
  const int wave = threadIdx.x >> 6, r = blockIdx.x * group_rows + wave;
  if (wave < group_rows && r < route_rows) {
    route_any(route, r, threadIdx.x & 63);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this row's ids (write-through stores) have reached memory before the ticket is drawn
  } else if (by_rows) {  // (one row a group) meanwhile, the wavefronts that route nothing
    constexpr int IDLE = PLAN_THREADS - 64;
    clear_plan(plan, slot_cap, blockIdx.x * IDLE + (int)threadIdx.x - 64, route_groups * IDLE);
  }
  __syncthreads();
  if (threadIdx.x == 0) last = last_to_arrive(plan, route_groups);
  __syncthreads();
  if (!last) return;  // the last arriver: every row's ids are in memory, and the plan reads them from there (load_through)
  if (by_rows) {
    plan_by_rows(ids, route_rows, route.k, e_lo, e_n, shared_rows, plan, order, slot_rows, slot_cap, lds, true);
  } else {
    plan_work<false>(ids, pairs, e_lo, e_n, shared_rows, plan, order, slot_rows, slot_cap, nullptr, 1, 0, 0, lds);
  }
}

// Budgeted selection and the plan of its ids in one launch: its workgroups rank `group_rows` rows each (a row a
// wavefront), and the last of them to finish selects and plans, as in the routing launch above: candidates and ids go through
// to memory, are waited for ahead of the ticket or the plan, and are read past the L2. (A rank launch of its own before it:
// 5.0 + 13.0 us at 40 rows of 512 experts, the whole layer 50.4 us and 48.7 so.) `PLAN`: false leaves the plan to launches of
// its own (more rows than plan_by_rows takes and PLACE_PAIRS pairs or more). `by_rows`: no row names an expert twice and they are at most
// PLAN_ROWS_MAX; each group ranks one.
template <int PER, bool PLAN>
__global__ __launch_bounds__(PLAN_THREADS) void moe_budget_plan_kernel(BudgetParams q, int copies_n, int e_lo, int e_n, int shared_rows,
                                                                       int32_t* __restrict__ plan, int32_t* __restrict__ order, int group_rows, int by_rows,
                                                                       int slot_rows, int slot_cap) {
  extern __shared__ int lds[];
  __shared__ int last;
  const int wave = threadIdx.x >> 6, r = blockIdx.x * group_rows + wave;
  if (wave < group_rows && r < q.r) {
    rank_row<PER, true>(q, r, threadIdx.x & 63);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  } else if (by_rows) {
    clear_plan(plan, slot_cap, blockIdx.x * (PLAN_THREADS - 64) + (int)threadIdx.x - 64, gridDim.x * (PLAN_THREADS - 64));
  }
  __syncthreads();
  if (threadIdx.x == 0) last = last_to_arrive(plan, gridDim.x);
  __syncthreads();
  if (!last) return;
  budget_pick<PER, false, true>(q, copies_n, reinterpret_cast<float*>(lds));
  if (!PLAN) return;
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wavefront's ids have reached memory
  __syncthreads();                                    // ... and everyone's; the selection's use of the LDS is over
  if (by_rows) {
    plan_by_rows(q.ids, q.r, q.k, e_lo, e_n, shared_rows, plan, order, slot_rows, slot_cap, lds, true);
  } else {
    plan_work<false>(q.ids, q.r * q.k, e_lo, e_n, shared_rows, plan, order, slot_rows, slot_cap, nullptr, 1, 0, 0, lds);
  }
}

// ---------------------------------------------------------------------------------------------------- combine
//
// out[r, c] = bf16( bf16(sum over the row's local slots, in selection order, of fma(w, y)) + g * shared ), one
// workgroup per (row, 512-column span). The reference's combine (hibana/kernels/csrc/w3_gemm.cu:1196-1213) when no
// shared expert is given; with one, its fused form (hibana/kernels/flashnext_fused.py:530-571).
constexpr int COMBINE_SPAN = 512;  // columns per workgroup (two per thread)

// A row's weighted sum of its pairs at columns c, c + 1, in selection order (FP32 fma chain). The pairs of B slots are
// read together (so the loads are all in flight at once) and a dropped slot contributes fma(0, 0, v).
template <int B, bool BF16>
struct CombineBatch {
  int e[B];
  float w[B];
  uint32_t half[B];
  float2 full[B];
  // every load of the batch is asked for before any is used: ids and weights (the same for the whole workgroup), then
  // the pairs - also a dropped slot's, whose values are then set aside (a pair's address does not depend on its id)
  __device__ __forceinline__ void load(const CombineParams& p, int r, int c, int s0) {
#pragma unroll
    for (int j = 0; j < B; j++) {
      const int s = min(s0 + j, p.topk - 1);
      e[j] = p.ids[r * p.topk + s];
      w[j] = p.weights[r * p.topk + s];
    }
#pragma unroll
    for (int j = 0; j < B; j++) {
      const int s = min(s0 + j, p.topk - 1);
      const int64_t at = ((int64_t)r * p.topk + s) * p.h + c;
      if (BF16) {
        half[j] = *reinterpret_cast<const uint32_t*>(reinterpret_cast<const uint16_t*>(p.pairs) + at);
      } else {
        full[j] = *reinterpret_cast<const float2*>(reinterpret_cast<const float*>(p.pairs) + at);
      }
    }
  }
  __device__ __forceinline__ void add(const CombineParams& p, int s0, float& v0, float& v1) {
    float y0[B], y1[B];
#pragma unroll
    for (int j = 0; j < B; j++) {
      const int local = e[j] - p.e_lo;
      const bool keep = s0 + j < p.topk && local >= 0 && local < p.e_n;
      const float a = BF16 ? __uint_as_float(half[j] << 16) : full[j].x, b = BF16 ? __uint_as_float(half[j] & 0xffff0000u) : full[j].y;
      y0[j] = keep ? a : 0.f;
      y1[j] = keep ? b : 0.f;
      w[j] = keep ? w[j] : 0.f;
    }
#pragma unroll
    for (int j = 0; j < B; j++) {
      v0 = fmaf(w[j], y0[j], v0);
      v1 = fmaf(w[j], y1[j], v1);
    }
  }
};

struct CombineShared {  // the shared expert's two columns, FP32 or BF16
  float2 f32 = {0.f, 0.f};
  uint32_t bf16 = 0;
  __device__ __forceinline__ void load(const CombineParams& p, int r, int c) {
    const int64_t at = (int64_t)r * p.shared_stride + c;
    if (p.shared_f32) {
      f32 = *reinterpret_cast<const float2*>(reinterpret_cast<const float*>(p.shared) + at);
    } else {
      bf16 = *reinterpret_cast<const uint32_t*>(reinterpret_cast<const uint16_t*>(p.shared) + at);
    }
  }
};

// One (row, 512-column span) a workgroup. The first batch of pairs and the shared expert's columns are asked for AHEAD
// of the gate's dot product, whose barrier would otherwise stand between two trips to memory: the gate's own loads
// follow them, and everything is on its way together.
template <int B, bool BF16>
__device__ __forceinline__ void combine_span(const CombineParams& p, float* red) {
  const int r = blockIdx.x;
  const int c = blockIdx.y * COMBINE_SPAN + 2 * threadIdx.x;  // h is even: a column pair is in or out together
  const bool in = c < p.h;                                    // a thread past the row's end reads column 0 and stores nothing: it is needed at the barrier
  const int cl = in ? c : 0;
  CombineBatch<B, BF16> batch;
  CombineShared sh;
  batch.load(p, r, cl, 0);
  if (p.shared) sh.load(p, r, cl);
  float g = 1.0f;
  if (p.gate_vec && p.shared) {  // uniform over the launch
    combine_gate_partial(p.x, p.gate_vec, p.hx, r, threadIdx.x, red);
    __syncthreads();
    g = combine_gate_value(red);
  }
  float v0 = 0.f, v1 = 0.f;
  batch.add(p, 0, v0, v1);
  for (int s0 = B; s0 < p.topk; s0 += B) {
    batch.load(p, r, cl, s0);
    batch.add(p, s0, v0, v1);
  }
  if (p.shared) {
    const float s0 = p.shared_f32 ? sh.f32.x : __uint_as_float(sh.bf16 << 16);
    const float s1 = p.shared_f32 ? sh.f32.y : __uint_as_float(sh.bf16 & 0xffff0000u);
    v0 = combine_shared(v0, g, s0);
    v1 = combine_shared(v1, g, s1);
  }
  if (in) *reinterpret_cast<uint32_t*>(p.out + (int64_t)r * p.h + c) = (uint32_t)f32_to_bf16_bits(v0) | ((uint32_t)f32_to_bf16_bits(v1) << 16);
}
// B: the slots read together - 8 or 12 where the call is long or top-k small, 24 for a short call of many slots
// (one wait on memory instead of three); a kernel of its own each, so that the longer batches' registers are theirs alone.
template <int B>
__global__ __launch_bounds__(256) void moe_combine_kernel(CombineParams p) {
  __shared__ float red[4];
  if (p.pairs_bf16) {
    combine_span<B, true>(p, red);
  } else {
    combine_span<B, false>(p, red);
  }
}

// A long call's sum of BF16 pairs alone: sixteen bytes of a pair a thread and load instead of four. combine_span's chain, operation
// for operation: the same bits. Bound by the pairs' traffic (5 TB/s). Measured alone, before and now: 1024 rows of 22 pairs, 1024
// columns, 12.7 and 10.8 us, 2048 rows 24.6 and 19.2; with the ids and weights asked for ahead of the pairs 9.0 and 15.7. (A row's ids
// and weights one at a time, behind its pairs, were a trip to memory each.)
template <int B>
__global__ __launch_bounds__(256) void moe_combine_wide_kernel(CombineParams p) {
  const int r = blockIdx.x, c = (blockIdx.y * blockDim.x + threadIdx.x) * 8;
  if (c >= p.h) return;  // h is a multiple of 8: a thread's columns are in or out together
  const uint16_t* at = static_cast<const uint16_t*>(p.pairs) + (int64_t)r * p.topk * p.h + c;
  float v[8];
#pragma unroll
  for (int i = 0; i < 8; i++) v[i] = 0.f;
  for (int s0 = 0; s0 < p.topk; s0 += B) {
    int e[B];
    float w[B];
    u32x4_t y[B];
#pragma unroll
    for (int j = 0; j < B; j++) {  // all asked for together
      e[j] = p.ids[r * p.topk + min(s0 + j, p.topk - 1)];
      w[j] = p.weights[r * p.topk + min(s0 + j, p.topk - 1)];
    }
#pragma unroll
    for (int j = 0; j < B; j++) y[j] = *reinterpret_cast<const u32x4_t*>(at + (int64_t)min(s0 + j, p.topk - 1) * p.h);
#pragma unroll
    for (int j = 0; j < B; j++) {
      const int local = e[j] - p.e_lo;
      const bool keep = s0 + j < p.topk && local >= 0 && local < p.e_n;
      const float weight = keep ? w[j] : 0.f;
#pragma unroll
      for (int i = 0; i < 8; i++) v[i] = fmaf(weight, keep ? (i & 1 ? pair_hi(y[j][i >> 1]) : pair_lo(y[j][i >> 1])) : 0.f, v[i]);
    }
  }
  u32x4_t out;
#pragma unroll
  for (int i = 0; i < 8; i += 2) out[i / 2] = (uint32_t)f32_to_bf16_bits(v[i]) | ((uint32_t)f32_to_bf16_bits(v[i + 1]) << 16);
  *reinterpret_cast<u32x4_t*>(p.out + (int64_t)r * p.h + c) = out;
}

// A row a workgroup, sixteen bytes of a pair a thread and load, the gate's dot product once a row: combine_span's chain and dot
// product, operation for operation: the same bits. There every span of 512 columns makes the dot product again, whose loads (12 KB
// at 2048 columns) are as many as the span's own. Bound by the pairs' traffic (3.7 TB/s at 1543 rows of 2048 columns). Measured alone, in spans
// and so, us, BF16, rows x pairs x columns: 1543 x 10 x 2048 22.8 and 15.3, x 1152 17.9 and 12.1, x 2304 (a second pass by 32 of 256 threads) 29.0
// and 22.5, x 2560 30.2 and 23.5; without a gate 21.1 and 13.9. Not below two spans of few pairs nor in one: 1543 x 6 x 1024 10.8 and 11.4, x 10
// x 1024 13.4 and 11.9, x 10 x 512 8.6 and 11.2. FP32 pairs, twice the registers and passes of the spans, only where four and more dot products
// are saved: 512 x 10 x 2048 10.9 and 10.4, 700 x 10 x 2560 18.0 and 16.3, 1000 x 12 x 2304 29.4 and 27.1, but 400 x 10 x 2048 9.3 and 9.6, 512 x 6 x
// 2048 8.7 and 9.2, 1000 x 6 x 1536 10.8 and 12.2, 700 x 10 x 2560 without a gate 14.2 and 15.9.
constexpr int COMBINE_ROW_FLOAT_ROWS = 512, COMBINE_ROW_FLOAT_COLUMNS = 4 * 512;
template <int B, bool BF16>
__global__ __launch_bounds__(256) void moe_combine_row_kernel(CombineParams p) {
  constexpr int V = BF16 ? 8 : 4;  // columns a load
  __shared__ float red[4];
  const int r = blockIdx.x;
  const uint8_t* pairs = static_cast<const uint8_t*>(p.pairs) + (int64_t)r * p.topk * p.h * (BF16 ? 2 : 4);
  const uint8_t* shared = static_cast<const uint8_t*>(p.shared) + (int64_t)r * p.shared_stride * (BF16 ? 2 : 4);
  float g = 1.0f;
  for (int c0 = 0; c0 < p.h; c0 += 256 * V) {
    const int c = c0 + V * threadIdx.x;
    const bool in = c < p.h;  // h is a multiple of 8
    const int at = in ? c * (BF16 ? 2 : 4) : 0;
    float v[V];
#pragma unroll
    for (int i = 0; i < V; i++) v[i] = 0.f;
    const u32x4_t sh = *reinterpret_cast<const u32x4_t*>(shared + at);
    for (int s0 = 0; s0 < p.topk; s0 += B) {
      int e[B];
      float w[B];
      u32x4_t y[B];
#pragma unroll
      for (int j = 0; j < B; j++) {
        e[j] = p.ids[r * p.topk + min(s0 + j, p.topk - 1)];
        w[j] = p.weights[r * p.topk + min(s0 + j, p.topk - 1)];
      }
#pragma unroll
      for (int j = 0; j < B; j++) y[j] = *reinterpret_cast<const u32x4_t*>(pairs + (int64_t)min(s0 + j, p.topk - 1) * p.h * (BF16 ? 2 : 4) + at);
      if (c0 == 0 && s0 == 0 && p.gate_vec) {  // uniform; behind the first loads, so that everything is on its way together
        combine_gate_partial(p.x, p.gate_vec, p.hx, r, threadIdx.x, red);
        __syncthreads();
        g = combine_gate_value(red);
      }
#pragma unroll
      for (int j = 0; j < B; j++) {
        const int local = e[j] - p.e_lo;
        const bool keep = s0 + j < p.topk && local >= 0 && local < p.e_n;
        const float weight = keep ? w[j] : 0.f;
#pragma unroll
        for (int i = 0; i < V; i++) v[i] = fmaf(weight, !keep ? 0.f : !BF16 ? __uint_as_float(y[j][i & 3]) : i & 1 ? pair_hi(y[j][i >> 1]) : pair_lo(y[j][i >> 1]), v[i]);
      }
    }
#pragma unroll
    for (int i = 0; i < V; i++) v[i] = combine_shared(v[i], g, !BF16 ? __uint_as_float(sh[i & 3]) : i & 1 ? pair_hi(sh[i >> 1]) : pair_lo(sh[i >> 1]));
    uint32_t out[V / 2];
#pragma unroll
    for (int i = 0; i < V; i += 2) out[i / 2] = (uint32_t)f32_to_bf16_bits(v[i]) | ((uint32_t)f32_to_bf16_bits(v[i + 1]) << 16);
    if (in) {
      if constexpr (BF16) {
        *reinterpret_cast<u32x4_t*>(p.out + (int64_t)r * p.h + c) = u32x4_t{out[0], out[1], out[2], out[3]};
      } else {
        *reinterpret_cast<uint2*>(p.out + (int64_t)r * p.h + c) = make_uint2(out[0], out[1]);
      }
    }
  }
}

// ------------------------------------------------------------------ the latent block's BF16 projections (M <= 16)
//
// y[i, n] = sum_k x[i, k] w[n, k] for at most sixteen rows of x, on the BF16 matrix cores with nothing staged: a
// wavefront takes sixteen weight rows over `steps` K steps of 32 from k0; lane (q, r16) holds k = 32 s + 8 q .. + 7 of
// weight row n0 + r16 (the B operand) and of activation row r16 (A; rows past m read row m - 1 and are never stored).
// Register i of lane (q, r16) of the result is y[4 q + i][n0 + r16]. Up to eight steps are in flight at a time.
struct GemvFrags {
  u32x4_t v[8];
};
__device__ __forceinline__ void gemv16_load(GemvFrags& f, const uint16_t* __restrict__ base, int64_t ld, int row, int k0, int steps, int lane) {
  const uint16_t* at = base + row * ld + k0 + 8 * (lane >> 4);
#pragma unroll
  for (int j = 0; j < 8; j++)
    if (j < steps) f.v[j] = *reinterpret_cast<const u32x4_t*>(at + 32 * j);
}
__device__ __forceinline__ void gemv16_mfma(f32x4_t& acc, const GemvFrags& a, const GemvFrags& b, int steps) {
#pragma unroll
  for (int j = 0; j < 8; j++)
    if (j < steps) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a.v[j]), __builtin_bit_cast(bf16x8_t, b.v[j]), acc, 0, 0, 0);
}
__device__ __forceinline__ f32x4_t gemv16_wave(const uint16_t* __restrict__ w, int64_t ldw, int n0, int n, const uint16_t* __restrict__ x, int64_t ldx, int m,
                                               int k0, int steps, int lane) {
  const int r16 = lane & 15, wrow = min(n0 + r16, n - 1), xrow = min(r16, m - 1);
  f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
  for (int s0 = 0; s0 < steps; s0 += 8) {
    GemvFrags a, b;
    gemv16_load(b, w, ldw, wrow, k0 + 32 * s0, steps - s0, lane);
    gemv16_load(a, x, ldx, xrow, k0 + 32 * s0, steps - s0, lane);
    gemv16_mfma(acc, a, b, steps - s0);
  }
  return acc;
}
// The K splits' partial tiles, one per wavefront, added in wavefront order: thread t < 256 returns y[t / 16][n0 + t % 16].
__device__ __forceinline__ float gemv16_reduce(const f32x4_t& acc, float* part, int waves) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  *reinterpret_cast<f32x4_t*>(part + wave * 256 + lane * 4) = acc;
  __syncthreads();
  float sum = 0.f;
  if (threadIdx.x < 256) {
    const int row = threadIdx.x >> 4, at = ((row >> 2) * 16 + (threadIdx.x & 15)) * 4 + (row & 3);
    for (int w = 0; w < waves; w++) sum += part[w * 256 + at];
  }
  return sum;
}

// The router's product of a routed layer for at most MOE_ROUTER_ROWS rows: latency bound (2 MB of weights), so sixteen
// columns and sixteen rows a workgroup and K over its sixteen wavefronts, every load of a wavefront's four steps in flight
// together. Partial tiles through LDS, added in wavefront order, rounded to BF16 once. At hidden 2048, 512 experts the
// library product it replaces took 8.4 - 8.7 us at 1, 32 and 40 rows, and another 2 us widened its BF16 result; the row
// tiles on one workgroup (sharing a weight fragment) 4.7, 7.9 and 9.6 us, on workgroups of their own 5.0, 5.8 and 6.0.
__global__ __launch_bounds__(1024) void moe_router_kernel(const uint16_t* __restrict__ w, const uint16_t* __restrict__ x, uint16_t* __restrict__ logits, int e,
                                                          int h, int m) {
  __shared__ __align__(16) float part[16 * 256];
  constexpr int BATCH = 4;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r16 = lane & 15, n0 = blockIdx.x * 16, m0 = blockIdx.y * 16;
  const int steps = h / 32, s0 = steps * wave / 16, s1 = steps * (wave + 1) / 16;
  const uint16_t* wat = w + (int64_t)min(n0 + r16, e - 1) * h + 8 * (lane >> 4);
  const uint16_t* xat = x + (int64_t)min(m0 + r16, m - 1) * h + 8 * (lane >> 4);
  f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
  for (int s = s0; s < s1; s += BATCH) {
    u32x4_t b[BATCH], a[BATCH];
#pragma unroll
    for (int j = 0; j < BATCH; j++)
      if (s + j < s1) {
        b[j] = *reinterpret_cast<const u32x4_t*>(wat + 32 * (s + j));
        a[j] = *reinterpret_cast<const u32x4_t*>(xat + 32 * (s + j));
      }
#pragma unroll
    for (int j = 0; j < BATCH; j++)
      if (s + j < s1) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a[j]), __builtin_bit_cast(bf16x8_t, b[j]), acc, 0, 0, 0);
  }
  *reinterpret_cast<f32x4_t*>(part + wave * 256 + lane * 4) = acc;
  __syncthreads();
  if (threadIdx.x < 256) {
    const int row = threadIdx.x >> 4, n = n0 + (threadIdx.x & 15), at = ((row >> 2) * 16 + (threadIdx.x & 15)) * 4 + (row & 3);
    float sum = 0.f;
#pragma unroll
    for (int v = 0; v < 16; v++) sum += part[v * 256 + at];
    if (m0 + row < m && n < e) logits[(int64_t)(m0 + row) * e + n] = bf16_of(sum);
  }
}

// The last launch of a small latent block (nemotron_moe.cu's out kernel): out = bf16(shared + routed fc2^T) with
// routed BF16 [m, latent]; sixteen output columns a workgroup, K split over its wavefronts (at most eight steps each).
struct OutGemv {
  const uint16_t* w;       // fc2 BF16 [n, k]
  const uint16_t* routed;  // BF16 [m, k]
  const uint16_t* shared;  // BF16 [m, n] or null
  uint16_t* out;           // BF16 [m, n]
  int n, k, m, waves;
};
__global__ __launch_bounds__(1024) void latent_out_kernel(OutGemv g) {
  __shared__ __align__(16) float part[16 * 256];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, n0 = blockIdx.x * 16;
  const int per_wave = g.k / g.waves;
  const int out_row = threadIdx.x >> 4, out_n = n0 + (threadIdx.x & 15);
  const bool stores = threadIdx.x < 256 && out_row < g.m && out_n < g.n;  // a workgroup has at least these 256 threads
  const float base = stores && g.shared ? bf16_bits_to_f32(g.shared[(int64_t)out_row * g.n + out_n]) : 0.f;
  f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
  if (wave < g.waves) acc = gemv16_wave(g.w, g.k, n0, g.n, g.routed, g.k, g.m, wave * per_wave, per_wave / 32, lane);
  const float sum = gemv16_reduce(acc, part, g.waves);
  if (stores) g.out[(int64_t)out_row * g.n + out_n] = f32_to_bf16_bits(base + sum);
}

// ---------------------------------------------------------------------------------------------------- host side
// The measurement hook's state: `g_events_armed` is all a launch reads while no events are armed (one relaxed load); the
// list itself is only touched under its lock.
static std::atomic<bool> g_events_armed{false};
static std::mutex g_events_lock;
static std::vector<hipEvent_t> g_events;
static size_t g_event_next = 0;
bool moe_next_events(hipEvent_t* start, hipEvent_t* stop) {
  if (!g_events_armed.load(std::memory_order_relaxed)) return false;
  std::lock_guard<std::mutex> hold(g_events_lock);
  if (g_event_next + 1 >= g_events.size()) return false;
  *start = g_events[g_event_next];
  *stop = g_events[g_event_next + 1];
  g_event_next += 2;
  return true;
}

void pick_shape(int n_blocks, int chunks, int64_t slots, int want, int* ks, int* nbw) {
  int k = 1;
  while (k < 16 && (int64_t)n_blocks * slots * k < want && chunks / (2 * k) >= 4) k *= 2;
  int b = k >= 4 ? 1 : 4 / k;
  while (b > 1 && n_blocks % b) b /= 2;
  *ks = k;
  *nbw = b;
}

int64_t moe_max_slots(int64_t pairs, int experts, int shared_rows, int slot_rows) {
  const int64_t routed = pairs < pairs / slot_rows + experts ? pairs : pairs / slot_rows + experts;
  return routed + (shared_rows + slot_rows - 1) / slot_rows;
}

static size_t align256(size_t v) { return (v + 255) & ~(size_t)255; }

MoeWorkspace moe_carve(void* base, int m, int topk, int experts, int inter, int hidden_out, int shared, int hidden) {
  const int64_t pairs = (int64_t)m * topk, rows = pairs + (shared ? m : 0);
  MoeWorkspace w{};
  size_t off = 0;
  auto take = [&](size_t bytes) {
    void* ptr = base ? static_cast<char*>(base) + off : nullptr;
    off += align256(bytes);
    return ptr;
  };
  w.plan = static_cast<int32_t*>(take((PLAN_HEADER + (4 + DONE_PITCH) * moe_max_slots(pairs, experts, shared ? m : 0, ROWS_PER_SLOT) + 32) * sizeof(int32_t)));  // entries, then plan_done
  w.plan_wide = static_cast<int32_t*>(take((size_t)PLAN_WIDE_GROUPS * experts * sizeof(int32_t)));
  w.order = static_cast<int32_t*>(take(rows * sizeof(int32_t)));
  w.h = static_cast<uint16_t*>(take((size_t)rows * inter * sizeof(uint16_t)));
  w.y = static_cast<float*>(take((size_t)rows * hidden_out * sizeof(float)));
  if (hidden) {
    w.xq = static_cast<uint8_t*>(take((size_t)m * hidden));
    w.xs = static_cast<float*>(take((size_t)m * (hidden / 32) * sizeof(float)));
    w.hq = static_cast<uint8_t*>(take((size_t)rows * inter));
    w.hs = static_cast<float*>(take((size_t)rows * (inter / 32) * sizeof(float)));
    w.x2 = static_cast<uint8_t*>(take((size_t)m * 2 * hidden));
    w.x2s = static_cast<float*>(take((size_t)m * sizeof(float)));
  }
  w.bytes = off;
  return w;
}

__global__ __launch_bounds__(256) void quant_groups_kernel(QuantJob job) {
  __shared__ float red[4];
  quant_job_share(job, blockIdx.x, red);
}

// BF16 [m, k] (k % 8 == 0) -> E4M3 codes [m, k] and ONE FP32 scale a row: s = max(amax / 448, 1e-12),
// q = e4m3(clamp(x / s, -448, 448)), IEEE divisions as in quant_groups_lane (the reference's per-row quantizer,
// hibana/kernels/csrc/w3_gemm.cu:244-288, which multiplies by a reciprocal). One workgroup a row: the row's largest
// magnitude over the four wavefronts through LDS, then every lane rounds its runs of eight values.
__global__ __launch_bounds__(256) void quant_rows_kernel(const uint16_t* __restrict__ x, int k, uint8_t* __restrict__ q, float* __restrict__ scales) {
  __shared__ float red[4];
  const int64_t row = blockIdx.x;
  const uint16_t* xr = x + row * k;
  float amax = 0.f;
  for (int c = 8 * threadIdx.x; c < k; c += 8 * 256) {
    const u32x4_t raw = *reinterpret_cast<const u32x4_t*>(xr + c);
#pragma unroll
    for (int j = 0; j < 4; j++) amax = fmaxf(amax, fmaxf(fabsf(__uint_as_float(raw[j] << 16)), fabsf(__uint_as_float(raw[j] & 0xffff0000u))));
  }
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) amax = fmaxf(amax, __shfl_xor(amax, d));
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = amax;
  __syncthreads();
  amax = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
  const float s = fmaxf(amax / 448.0f, 1e-12f);
  if (threadIdx.x == 0) scales[row] = s;
  for (int c = 8 * threadIdx.x; c < k; c += 8 * 256) {
    const u32x4_t raw = *reinterpret_cast<const u32x4_t*>(xr + c);
    float v[8];
#pragma unroll
    for (int j = 0; j < 4; j++) {
      v[2 * j] = __uint_as_float(raw[j] << 16);
      v[2 * j + 1] = __uint_as_float(raw[j] & 0xffff0000u);
    }
#pragma unroll
    for (int j = 0; j < 8; j++) v[j] = fminf(fmaxf(v[j] / s, -448.0f), 448.0f);
    int lo = 0, hi = 0;
    lo = __builtin_amdgcn_cvt_pk_fp8_f32(v[0], v[1], lo, false);
    lo = __builtin_amdgcn_cvt_pk_fp8_f32(v[2], v[3], lo, true);
    hi = __builtin_amdgcn_cvt_pk_fp8_f32(v[4], v[5], hi, false);
    hi = __builtin_amdgcn_cvt_pk_fp8_f32(v[6], v[7], hi, true);
    typedef __attribute__((ext_vector_type(2))) int i32x2_t;
    *reinterpret_cast<i32x2_t*>(q + row * k + c) = i32x2_t{lo, hi};
  }
}

void moe_launch_quant_rows(const uint16_t* x, int64_t m, int k, uint8_t* q, float* scales, hipStream_t stream) {
  HB_LAUNCH(quant_rows_kernel, dim3((unsigned)m), dim3(256), 0, stream, x, k, q, scales);
}

void moe_launch_quant_groups(const QuantJob& job, hipStream_t stream) {
  const unsigned groups = job.split_rows ? (unsigned)job.split_rows : (unsigned)((job.lanes + 255) / 256);
  HB_LAUNCH(quant_groups_kernel, dim3(groups), dim3(256), 0, stream, job);
}

static std::atomic<int> g_route_plan_fused{0};  // hb_tune("route_plan", 2): routing and plan as two launches; 1: the general plan also where plan_by_rows serves
static std::atomic<int> g_fault_inject{0};
int moe_tune(const char* key, int value) {
  if (!strcmp(key, "fault_inject") && (value == 0 || value == 1)) {
    g_fault_inject.store(value, std::memory_order_relaxed);
    return HB_OK;
  }
  if (strcmp(key, "route_plan") || value < 0 || value > 2) return HB_EINVAL;
  g_route_plan_fused.store(value, std::memory_order_relaxed);
  return HB_OK;
}

void moe_await_slots(StreamParams& p1, StreamParams& p2, int32_t* plan, int64_t slots, int groups1) {
  const bool inject = g_fault_inject.load(std::memory_order_relaxed) == 1;  // a test of the give-up path: a count one above what can arrive, a wait of a few polls
  p1.done = p2.done = plan_done(plan, slots);
  p1.done_need = p2.done_need = groups1 + (inject ? 1 : 0);
  p2.wait_spins = inject ? 8 : WAIT_SPINS;
  p2.fault = plan + PLAN_FAULT;
}

// From this many pairs: the layer of 65 and 80 rows of ten took 66.5 and 71.8 us with one workgroup, 67.1 and 72.5 in shares, of 128
// rows 80.8 and 77.9, of 256 rows 113.6 and 108.8; a latent block of 64 rows of 22 283 and 278. Under a budget (the plan behind the selection in
// its launch, and in shares): 96 rows of ten 74.7 and 75.0, 104 79.9 and 79.0, 128 83.3 and 82.4, 400 157.3 and 151.7; of 96 experts (1024, 256) 104
// rows 50.2 and 50.5, 128 52.8 and 52.9, 256 74.0 and 72.3.
constexpr int64_t PLACE_PAIRS = 1024;
static unsigned plan_groups(const QuantJob* job) {
  if (!job) return 1u;
  return 1u + (job->split_rows ? (unsigned)job->split_rows : (unsigned)((job->lanes + PLAN_THREADS - 1) / PLAN_THREADS));
}

int moe_launch_plan(const int32_t* ids, int64_t pairs, int e_lo, int e_n, int shared_rows, const MoeWorkspace& ws, hipStream_t stream, int slot_rows,
                    const QuantJob* job, int distinct) {
  const size_t plan_lds = ((size_t)(PLAN_WAVES + 1) * e_n + 3 * (PLAN_WAVES + 1)) * sizeof(int);
  if (plan_lds > 64 * 1024 || e_n > PLAN_THREADS || pairs > 0x3fffffff) return HB_EINVAL;
  const int slot_cap = (int)moe_max_slots(pairs, distinct ? distinct : e_n, shared_rows, slot_rows);
  if (!job && pairs >= PLACE_PAIRS && pairs <= PLACE_TABLE_SHARE * PLAN_WIDE_GROUPS) {
    auto place = [&](auto kernel, int share, int tiles) {
      const size_t lds = ((size_t)tiles * e_n + 3 * (PLAN_WAVES + 1)) * sizeof(int);
      HB_LAUNCH(kernel, dim3((unsigned)((pairs + share - 1) / share)), dim3(PLAN_THREADS), lds, stream, ids, (int)pairs, e_lo, e_n, shared_rows, ws.plan,
                ws.order, slot_rows, slot_cap, ws.plan_wide);
    };
    if (pairs < PLAN_WIDE_PAIRS) {
      place(moe_place_kernel<false>, PLACE_SHARE, PLACE_SHARE / 64 + 2);
    } else {
      const int groups = (int)((pairs + PLACE_TABLE_SHARE - 1) / PLACE_TABLE_SHARE);  // the counting workgroups' shares are the placing ones'
      HB_LAUNCH(moe_plan_kernel<true>, dim3(groups), dim3(PLAN_THREADS), plan_lds, stream, ids, (int)pairs, e_lo, e_n, shared_rows, ws.plan, ws.order,
                RouteParams{}, 0, 0, slot_rows, slot_cap, ws.plan_wide, groups, 1, QuantJob{});
      place(moe_place_kernel<true>, PLACE_TABLE_SHARE, PLACE_TABLE_SHARE / 64);
    }
    return HB_OK;
  }
  if (pairs >= PLAN_WIDE_PAIRS) {  // a share of about a thousand pairs a workgroup
    const int groups = (int)std::min<int64_t>(PLAN_WIDE_GROUPS, pairs / 1024);
    if (job) moe_launch_quant_groups(*job, stream);
    for (int phase = 1; phase <= 3; phase++)
      HB_LAUNCH(moe_plan_kernel<true>, dim3(phase == 2 ? 1 : groups), dim3(PLAN_THREADS), plan_lds, stream, ids, (int)pairs, e_lo, e_n, shared_rows, ws.plan,
                ws.order, RouteParams{}, 0, 0, slot_rows, slot_cap, ws.plan_wide, groups, phase, QuantJob{});
    return HB_OK;
  }
  HB_LAUNCH(moe_plan_kernel<false>, dim3(plan_groups(job)), dim3(PLAN_THREADS), plan_lds, stream, ids, (int)pairs, e_lo, e_n, shared_rows, ws.plan, ws.order,
            RouteParams{}, 0, 0, slot_rows, slot_cap, ws.plan_wide, 1, 0, job ? *job : QuantJob{});
  return HB_OK;
}

int moe_check_route(int m, int e, int k) { return m <= 0 || e <= 0 || k <= 0 || k > e || k > 64 || e > 64 * ROUTE_PER_LANE ? HB_EINVAL : HB_OK; }

// From more rows than compute units a workgroup routes several: each is a full one, of which a compute unit holds two, and all
// draw tickets from one counter. So many rows come here with E4M3 activations (whose rounding rides in the launch) or few selections: the
// E4M3 layer of 512 experts, rows of ten, a row, eight and sixteen rows a workgroup, 300 rows 206.1, 201.5 and 202.4 us, 400 rows 223.0, 218.0
// and 219.6, 800 rows 329.0, 317.9 and 318.1; weight-only, rows of three, 300 rows 138.9, 135.2 and 135.9.
constexpr int ROUTE_GROUP_ROWS = 8, ROUTE_SPREAD_ROWS = 256;
// Whether no row names an expert twice: every row is real, or a padded row names none (with `repeat` it names one over and over).
static bool rows_distinct(const RouteParams& rp, int e_lo, int e_n) { return !rp.slots || (!rp.repeat && (rp.pad_id < e_lo || rp.pad_id >= e_lo + e_n)); }
// Routing by `rp` (either rule) and the plan of its ids, in as few launches as the size allows.
static int launch_route_plan(const RouteParams& rp, int m, int e_lo, int e_n, int shared_rows, const MoeWorkspace& ws, hipStream_t stream, int slot_rows,
                             const QuantJob* job) {
  const int64_t pairs = (int64_t)m * rp.k;
  const size_t plan_lds = ((size_t)(PLAN_WAVES + 1) * e_n + 3 * (PLAN_WAVES + 1)) * sizeof(int);
  if (plan_lds > 64 * 1024 || e_n > PLAN_THREADS || pairs > 0x3fffffff) return HB_EINVAL;
  const int by_rows = rows_distinct(rp, e_lo, e_n) && m <= PLAN_ROWS_MAX && rp.k <= 64 && g_route_plan_fused.load(std::memory_order_relaxed) != 1;
  const bool apart = !job && m > PLAN_ROWS_MAX && pairs >= PLACE_PAIRS && g_route_plan_fused.load(std::memory_order_relaxed) == 0;
  if (m > ROUTE_FUSED_ROWS && pairs < PLAN_WIDE_PAIRS && g_route_plan_fused.load(std::memory_order_relaxed) != 2 && !apart) {
    // a verify-sized call: the routing spread over the device, the plan by the workgroup that finishes last
    const int group_rows = m <= ROUTE_SPREAD_ROWS ? 1 : ROUTE_GROUP_ROWS, groups = (m + group_rows - 1) / group_rows;
    HB_LAUNCH(moe_route_plan_kernel, dim3((unsigned)groups + plan_groups(job) - 1u), dim3(PLAN_THREADS), plan_lds, stream, rp.ids, (int)pairs, e_lo, e_n,
              shared_rows, ws.plan, ws.order, rp, m, groups, group_rows, by_rows, slot_rows, (int)moe_max_slots(pairs, e_n, shared_rows, slot_rows),
              job ? *job : QuantJob{});
    return HB_OK;
  }
  if (m > ROUTE_FUSED_ROWS) {  // a prefill-sized call: a wavefront a row over the whole device, then the plan's launches
    if (rp.sigmoid) {
      launch_route<true>(rp, m, stream);
    } else {
      launch_route<false>(rp, m, stream);
    }
    return moe_launch_plan(rp.ids, pairs, e_lo, e_n, shared_rows, ws, stream, slot_rows, job);
  }
  static_assert(ROUTE_FUSED_ROWS <= PLAN_WAVES, "a wavefront a row");
  HB_LAUNCH(moe_plan_kernel<false>, dim3(plan_groups(job)), dim3(PLAN_THREADS), plan_lds, stream, rp.ids, (int)pairs, e_lo, e_n, shared_rows, ws.plan, ws.order,
            rp, m, by_rows && pairs > ROUTE_FEW_PAIRS, slot_rows, (int)moe_max_slots(pairs, e_n, shared_rows, slot_rows),
            ws.plan_wide, 1, 0, job ? *job : QuantJob{});
  return HB_OK;
}

void moe_launch_router(const uint16_t* x, const uint16_t* w, int m, int e, int h, uint16_t* logits, hipStream_t stream) {
  HB_LAUNCH(moe_router_kernel, dim3((unsigned)((e + 15) / 16), (unsigned)((m + 15) / 16)), dim3(1024), 0, stream, w, x, logits, e, h, m);
}

int moe_launch_route_plan(const TopkRoute& route, int m, int topk, int32_t* ids, float* weights, int e_lo, int e_n, int shared_rows,
                          const MoeWorkspace& ws, hipStream_t stream, int slot_rows, const QuantJob* job) {
  if (int err = moe_check_route(m, route.e, topk)) return err;
  RouteParams rp{};
  rp.logits = static_cast<const float*>(route.logits);
  rp.half = route.half;
  rp.stride = route.e;
  rp.slots = route.slots;
  rp.e = route.e;
  rp.k = topk;
  rp.per = (route.e + 63) / 64;
  rp.steps = route.steps;
  rp.pad_id = route.e;
  rp.ids = ids;
  rp.weights = weights;
  return launch_route_plan(rp, m, e_lo, e_n, shared_rows, ws, stream, slot_rows, job);
}

int moe_check_budget(const BudgetRoute& b, int m, int topk) {
  const bool refused = b.e < BUDGET_CANDIDATES || b.e > BUDGET_THREADS || topk > BUDGET_CANDIDATES || b.keep < 0 || b.keep > BUDGET_CANDIDATES || b.budget < 0 ||
                       b.steps <= 0 || m % b.steps || b.per_request < 0 || b.min_cap < 0 || !aligned(b.logits, 2) || !aligned(b.slots, 4);
  return refused ? HB_EINVAL : HB_OK;
}

constexpr int BUDGET_SPREAD_ROWS = 256;  // about the compute units
int moe_launch_budget_plan(const BudgetRoute& b, int m, int topk, int32_t* ids, float* weights, int e_lo, int e_n, int shared_rows,
                           const MoeWorkspace& ws, void* scratch, hipStream_t stream, int slot_rows) {
  static_assert(BUDGET_THREADS == PLAN_THREADS, "the selection and the plan share a workgroup");
  const int64_t pairs = (int64_t)m * topk;
  const size_t plan_lds = ((size_t)(PLAN_WAVES + 1) * e_n + 3 * (PLAN_WAVES + 1)) * sizeof(int);
  if (plan_lds > 64 * 1024 || e_n > PLAN_THREADS || pairs > 0x3fffffff) return HB_EINVAL;
  if (!b.logits || !scratch) return HB_ENULL;
  if (!aligned(scratch, 4)) return HB_EINVAL;
  if (int e = moe_check_budget(b, m, topk)) return e;
  BudgetParams q{};
  q.logits = b.logits;
  q.slots = b.slots;
  q.r = m, q.e = b.e, q.k = topk, q.keep = b.keep, q.budget = b.budget, q.per_request = b.per_request, q.min_cap = b.min_cap, q.steps = b.steps,
  q.repeat = b.repeat;
  q.cands = BUDGET_CANDIDATES;
  q.cand = static_cast<int32_t*>(scratch);
  q.prob = reinterpret_cast<float*>(q.cand + (int64_t)m * BUDGET_CANDIDATES);
  q.share = q.prob;
  q.ids = ids, q.weights = weights;
  const bool small = b.e <= 512;
  const int copies_n = small ? BUDGET_WAVES : BUDGET_WAVES / 2;
  const size_t pick_lds = (size_t)copies_n * b.e * sizeof(float);
  const int distinct = (int)budget_distinct(b, m, e_n), slot_cap = (int)moe_max_slots(pairs, distinct, shared_rows, slot_rows);
  const bool plan = m <= PLAN_ROWS_MAX || pairs < PLACE_PAIRS, by_rows = plan && !b.repeat && m <= PLAN_ROWS_MAX && topk <= 64;
  const int group_rows = m <= BUDGET_SPREAD_ROWS ? 1 : PLAN_WAVES;  // a row a workgroup while that spreads them over the device
  const dim3 grid((unsigned)((m + group_rows - 1) / group_rows));
  const size_t lds = plan ? std::max(pick_lds, plan_lds) : pick_lds;
  auto launch = [&](auto kernel) {
    HB_LAUNCH(kernel, grid, dim3(PLAN_THREADS), lds, stream, q, copies_n, e_lo, e_n, shared_rows, ws.plan, ws.order, group_rows, (int)by_rows, slot_rows,
              slot_cap);
  };
  if (plan) {
    small ? launch(moe_budget_plan_kernel<8, true>) : launch(moe_budget_plan_kernel<16, true>);
    return HB_OK;
  }
  small ? launch(moe_budget_plan_kernel<8, false>) : launch(moe_budget_plan_kernel<16, false>);
  return moe_launch_plan(ids, pairs, e_lo, e_n, shared_rows, ws, stream, slot_rows, nullptr, distinct);
}

static RouteParams latent_route(const LatentRouter& r) {
  RouteParams rp{};
  rp.sigmoid = 1;
  rp.logits = r.fused;
  rp.stride = r.experts + r.latent;
  rp.bias = r.bias;
  rp.slots = r.slots;
  rp.steps = r.steps;
  rp.repeat = r.pad_id < 0;
  rp.pad_id = r.pad_id;
  rp.e = r.experts;
  rp.k = r.topk;
  rp.per = (r.experts + 63) / 64;
  rp.latent = r.latent;
  rp.ids = r.ids;
  rp.weights = r.weights;
  rp.lat = nullptr;  // the product's epilogue has written them
  return rp;
}

int latent_launch_route(const LatentRouter& r, hipStream_t stream) {
  if (int err = moe_check_route(r.m, r.experts, r.topk)) return err;
  const RouteParams rp = latent_route(r);
  if (!r.ws) {  // no plan to fill: the routing alone
    launch_route<true>(rp, r.m, stream);
    return HB_OK;
  }
  return launch_route_plan(rp, r.m, r.e_lo, r.e_n, 0, *r.ws, stream, ROWS_PER_SLOT, nullptr);
}

bool latent_plan_of(const LatentRouter& r, LatentPlan& q) {
  const int64_t pairs = (int64_t)r.m * r.topk;
  q.lds = ((size_t)(PLAN_WAVES + 1) * r.e_n + 3 * (PLAN_WAVES + 1)) * sizeof(int);
  if (!r.ws || q.lds > 64 * 1024 || r.e_n > PLAN_THREADS || g_route_plan_fused.load(std::memory_order_relaxed) != 0) return false;
  q.route = latent_route(r);
  q.groups = r.m <= ROUTE_FUSED_ROWS ? 1 : r.m;
  q.by_rows = rows_distinct(q.route, r.e_lo, r.e_n) && r.topk <= 64 && (q.groups > 1 || pairs > ROUTE_FEW_PAIRS);
  q.slot_cap = (int)moe_max_slots(pairs, r.e_n, 0, ROWS_PER_SLOT);
  return true;
}

int latent_launch_out(const uint16_t* fc2, const uint16_t* routed, const uint16_t* shared, uint16_t* out, int m, int hidden, int latent, hipStream_t stream) {
  if (m <= 0 || m > LATENT_MAX_ROWS || hidden <= 0 || latent <= 0 || latent % 32) return HB_EINVAL;
  const int steps = latent / 32;
  int waves = 1;
  while (waves < 16 && (steps % waves || steps / waves > 8)) waves *= 2;
  if (steps % waves || steps / waves > 8) return HB_EINVAL;
  OutGemv g{fc2, routed, shared, out, hidden, latent, m, waves};
  HB_LAUNCH(latent_out_kernel, dim3((unsigned)((hidden + 15) / 16)), dim3((unsigned)std::max(256, 64 * waves)), 0, stream, g);
  return HB_OK;
}

void moe_launch_combine(const CombineParams& c, hipStream_t stream) {
  // the wide form from the size that its comment measures (a summed call's pairs are FP32 below), where the addresses allow it
  if (c.pairs_bf16 && !c.shared && c.m >= MOE_WIDE_ROWS && c.h % 8 == 0 && aligned(c.pairs, 16) && aligned(c.out, 16)) {
    const int threads = std::min(256, (c.h / 8 + 63) / 64 * 64);
    HB_LAUNCH(moe_combine_wide_kernel<12>, dim3((unsigned)c.m, (unsigned)((c.h / 8 + threads - 1) / threads)), dim3((unsigned)threads), 0, stream, c);
    return;
  }
  // ... and with a shared expert a row a workgroup, by the lines that its comment measures
  const bool many = c.topk > 8;
  const bool row = c.pairs_bf16 ? c.m >= MOE_WIDE_ROWS && (c.h > 2 * COMBINE_SPAN || (c.h > COMBINE_SPAN && many))
                                : c.m >= COMBINE_ROW_FLOAT_ROWS && c.h >= COMBINE_ROW_FLOAT_COLUMNS && many && c.gate_vec;
  if (c.shared && row && c.h % 8 == 0 && c.shared_stride % 8 == 0 && (c.pairs_bf16 != 0) == (c.shared_f32 == 0) && aligned(c.pairs, 16) && aligned(c.shared, 16) &&
      aligned(c.out, 16)) {
    if (c.pairs_bf16) {
      HB_LAUNCH((moe_combine_row_kernel<12, true>), dim3((unsigned)c.m), dim3(256), 0, stream, c);
    } else {
      HB_LAUNCH((moe_combine_row_kernel<12, false>), dim3((unsigned)c.m), dim3(256), 0, stream, c);
    }
    return;
  }
  const dim3 grid((unsigned)c.m, (unsigned)((c.h + COMBINE_SPAN - 1) / COMBINE_SPAN));
  if (c.topk <= 8 || (c.topk > 12 && c.m > 64)) {  // a long call is bound by its traffic: fewer registers, more wavefronts
    HB_LAUNCH(moe_combine_kernel<8>, grid, dim3(256), 0, stream, c);
  } else if (c.topk <= 12) {
    HB_LAUNCH(moe_combine_kernel<12>, grid, dim3(256), 0, stream, c);
  } else {
    HB_LAUNCH(moe_combine_kernel<24>, grid, dim3(256), 0, stream, c);
  }
}

}  // namespace hb

using namespace hb;

extern "C" int hb_moe_combine_pairs(const void* pairs, int pairs_bf16, const int32_t* ids, const float* weights, const void* shared,
                                    const void* x, const float* gate_vec, int e_lo, int e_n, int m, int topk, int h, void* out,
                                    void* stream) {
  if (!pairs || !ids || !weights || !out) return HB_ENULL;
  if (gate_vec && shared && !x) return HB_ENULL;
  if (m <= 0 || topk <= 0 || h <= 0 || h % 2) return HB_EINVAL;
  if (!aligned(pairs, 8) || !aligned(ids, 4) || !aligned(weights, 4) || !aligned(shared, 4) || !aligned(x, 2) || !aligned(gate_vec, 4) || !aligned(out, 4))
    return HB_EINVAL;
  CombineParams c{};
  c.pairs = pairs;
  c.pairs_bf16 = pairs_bf16;
  c.ids = ids;
  c.weights = weights;
  c.shared = shared;
  c.shared_stride = h;
  c.x = static_cast<const uint16_t*>(x);
  c.gate_vec = gate_vec;
  c.hx = h;
  c.e_lo = e_lo;
  c.e_n = e_n;
  c.m = m;
  c.topk = topk;
  c.h = h;
  c.out = static_cast<uint16_t*>(out);
  moe_launch_combine(c, as_stream(stream));
  return launch_status();
}

// out[r, c] = bf16( bf16(silu(gate)) * up ) of BF16 rows holding `half` gate and `half` up columns: [gate | up]
// (pairs == 0) or alternating blocks of `pairs` gate columns and their `pairs` up columns. The roundings are those of
// the BF16 tensor expression silu(gate) * up (hibana/kernels/ops.py:86-92 of the reference); without CHAIN the FP32
// product is rounded once. Two columns a thread.
template <bool CHAIN>
__global__ __launch_bounds__(256) void silu_and_mul_kernel(const uint16_t* __restrict__ x, int64_t rows, int half, int pairs, uint16_t* __restrict__ out) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;  // column pair i % (half / 2) of row i / (half / 2)
  const int per_row = half >> 1;
  if (i >= rows * per_row) return;
  const int64_t r = i / per_row;
  const int c = 2 * (int)(i - r * per_row);
  const int gate_at = pairs ? (c / pairs) * 2 * pairs + c % pairs : c, up_at = pairs ? gate_at + pairs : half + c;
  const uint16_t* row = x + r * 2 * half;
  const uint32_t g2 = *reinterpret_cast<const uint32_t*>(row + gate_at), u2 = *reinterpret_cast<const uint32_t*>(row + up_at);
  const float g0 = __uint_as_float(g2 << 16), g1 = __uint_as_float(g2 & 0xffff0000u);
  const float u0 = __uint_as_float(u2 << 16), u1 = __uint_as_float(u2 & 0xffff0000u);
  float s0 = g0 / (1.0f + expf(-g0)), s1 = g1 / (1.0f + expf(-g1));
  if (CHAIN) s0 = round_bf16(s0), s1 = round_bf16(s1);
  *reinterpret_cast<uint32_t*>(out + r * half + c) = (uint32_t)f32_to_bf16_bits(s0 * u0) | ((uint32_t)f32_to_bf16_bits(s1 * u1) << 16);
}

static int silu_mul_launch(const void* gate_up, int64_t rows, int half, int pairs, bool chain, void* out, void* stream) {
  if (!gate_up || !out) return HB_ENULL;
  if (rows <= 0 || half <= 0 || half % 2 || pairs < 0 || (pairs && (pairs % 2 || half % pairs))) return HB_EINVAL;
  if (!aligned(gate_up, 4) || !aligned(out, 4)) return HB_EINVAL;
  const int64_t threads = rows * (half / 2);
  const dim3 grid((unsigned)((threads + 255) / 256));
  if (chain) {
    hipLaunchKernelGGL(silu_and_mul_kernel<true>, grid, dim3(256), 0, as_stream(stream), static_cast<const uint16_t*>(gate_up), rows, half, pairs,
                       static_cast<uint16_t*>(out));
  } else {
    hipLaunchKernelGGL(silu_and_mul_kernel<false>, grid, dim3(256), 0, as_stream(stream), static_cast<const uint16_t*>(gate_up), rows, half, pairs,
                       static_cast<uint16_t*>(out));
  }
  return launch_status();
}

extern "C" int hb_silu_and_mul(const void* gate_up, int64_t rows, int half, int pairs, void* out, void* stream) {
  return silu_mul_launch(gate_up, rows, half, pairs, true, out, stream);
}

// bf16(silu(gate) * up) from the FP32 product: one rounding (silu_mul, hibana/kernels/flashnext_fused.py:624-639).
extern "C" int hb_silu_mul(const void* gate_up, int64_t rows, int half, int pairs, void* out, void* stream) {
  return silu_mul_launch(gate_up, rows, half, pairs, false, out, stream);
}

// (q, scales) = the per-(row, 32-group) E4M3 rounding of silu(gate) * up in one launch: BF16 [rows, 2 half] with the
// gate | up columns as in silu_and_mul_kernel -> E4M3 [rows, half], FP32 scales [rows, half / 32]. The product is
// rounded to BF16 as that kernel does it (`torch_chain`: silu to BF16 first, then the BF16 product) or from the FP32
// product with one rounding; the rounding to E4M3 is quant_groups_lane's, value for value (silu_mul_quant_groups,
// hibana/kernels/flashnext_fused.py:814-853 of the reference, with the exact divisions of its torch statement). A lane
// takes eight consecutive output columns, four lanes a group.
__global__ __launch_bounds__(256) void silu_mul_quant_groups_kernel(const uint16_t* __restrict__ x, int64_t rows, int half, int pairs, int torch_chain,
                                                                    uint8_t* __restrict__ q, float* __restrict__ scales) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;  // eight columns from 8 (i % (half / 8)) of row i / (half / 8)
  const int per_row = half >> 3;
  if (i >= rows * per_row) return;  // whole groups leave together: rows * per_row is a multiple of four
  const int64_t r = i / per_row;
  const int c = 8 * (int)(i - r * per_row);
  const int gate_at = pairs ? (c / pairs) * 2 * pairs + c % pairs : c, up_at = pairs ? gate_at + pairs : half + c;
  const uint16_t* row = x + r * 2 * half;
  const u32x4_t g4 = *reinterpret_cast<const u32x4_t*>(row + gate_at), u4 = *reinterpret_cast<const u32x4_t*>(row + up_at);
  float v[8];
#pragma unroll
  for (int j = 0; j < 8; j++) {
    const float g = __uint_as_float((j & 1) ? g4[j >> 1] & 0xffff0000u : g4[j >> 1] << 16);
    const float u = __uint_as_float((j & 1) ? u4[j >> 1] & 0xffff0000u : u4[j >> 1] << 16);
    v[j] = torch_chain ? silu_chain(g, u) : round_bf16(g / (1.0f + expf(-g)) * u);
  }
  float amax = 0.f;
#pragma unroll
  for (int j = 0; j < 8; j++) amax = fmaxf(amax, fabsf(v[j]));
  amax = fmaxf(amax, __shfl_xor(amax, 1));
  amax = fmaxf(amax, __shfl_xor(amax, 2));
  const float s = fmaxf(amax / 448.0f, 1e-12f);
#pragma unroll
  for (int j = 0; j < 8; j++) v[j] = fminf(fmaxf(v[j] / s, -448.0f), 448.0f);
  int lo = 0, hi = 0;
  lo = __builtin_amdgcn_cvt_pk_fp8_f32(v[0], v[1], lo, false);
  lo = __builtin_amdgcn_cvt_pk_fp8_f32(v[2], v[3], lo, true);
  hi = __builtin_amdgcn_cvt_pk_fp8_f32(v[4], v[5], hi, false);
  hi = __builtin_amdgcn_cvt_pk_fp8_f32(v[6], v[7], hi, true);
  typedef __attribute__((ext_vector_type(2))) int i32x2_t;
  *reinterpret_cast<i32x2_t*>(q + r * half + c) = i32x2_t{lo, hi};
  if ((c & 31) == 0) scales[r * (half >> 5) + (c >> 5)] = s;
}

extern "C" int hb_silu_mul_quant_groups(const void* gate_up, int64_t rows, int half, int pairs, int torch_chain, void* q, float* scales, void* stream) {
  if (!gate_up || !q || !scales) return HB_ENULL;
  if (rows <= 0 || half <= 0 || half % 32 || pairs < 0 || (pairs && (pairs % 32 || half % pairs))) return HB_EINVAL;
  if (!aligned(gate_up, 16) || !aligned(q, 8) || !aligned(scales, 4)) return HB_EINVAL;
  const int64_t threads = rows * (half / 8);
  hipLaunchKernelGGL(silu_mul_quant_groups_kernel, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, as_stream(stream),
                     static_cast<const uint16_t*>(gate_up), rows, half, pairs, torch_chain, static_cast<uint8_t*>(q), scales);
  return launch_status();
}

// x[r, c] = bf16(relu(x[r, c])^2) in place for BF16 rows `stride` elements apart: the square in FP32, one rounding
// (torch's relu(x) ** 2; relu2_, hibana/model/nemotron/moe.py:316-321 of the reference). Two columns a thread.
__global__ __launch_bounds__(256) void relu2_kernel(uint16_t* __restrict__ x, int64_t rows, int n, int64_t stride) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int per_row = n >> 1;
  if (i >= rows * per_row) return;
  const int64_t r = i / per_row;
  uint32_t* at = reinterpret_cast<uint32_t*>(x + r * stride + 2 * (i - r * per_row));
  const uint32_t two = *at;
  const float a = fmaxf(__uint_as_float(two << 16), 0.f), b = fmaxf(__uint_as_float(two & 0xffff0000u), 0.f);
  *at = (uint32_t)f32_to_bf16_bits(a * a) | ((uint32_t)f32_to_bf16_bits(b * b) << 16);
}

extern "C" int hb_relu2(void* x, int64_t rows, int n, int64_t stride, void* stream) {
  if (!x) return HB_ENULL;
  if (rows <= 0 || n <= 0 || n % 2 || stride < n || stride % 2) return HB_EINVAL;
  if (!aligned(x, 4)) return HB_EINVAL;
  const int64_t threads = rows * (n / 2);
  hipLaunchKernelGGL(relu2_kernel, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, as_stream(stream), static_cast<uint16_t*>(x), rows, n, stride);
  return launch_status();
}

extern "C" int hb_route_softmax_topk(const float* logits, int m, int e, int k, const int32_t* slots, int steps, int repeat, int32_t* ids,
                                     float* weights, void* stream) {
  if (!logits || !ids || !weights) return HB_ENULL;
  if (m <= 0 || e <= 0 || k <= 0 || k > e || k > 64 || e > 64 * ROUTE_PER_LANE || steps <= 0) return HB_EINVAL;
  if (!aligned(logits, 4) || !aligned(slots, 4) || !aligned(ids, 4) || !aligned(weights, 4)) return HB_EINVAL;
  RouteParams p{};
  p.logits = logits;
  p.stride = e;
  p.slots = slots;
  p.steps = steps;
  p.repeat = repeat;
  p.e = e;
  p.k = k;
  p.per = (e + 63) / 64;
  p.pad_id = e;
  p.ids = ids;
  p.weights = weights;
  launch_route<false>(p, m, as_stream(stream));
  return launch_status();
}

extern "C" int hb_route_sigmoid_topk(const float* fused, int64_t stride, const float* bias, int m, int e, int k, int latent,
                                     const int32_t* slots, int steps, int repeat, int32_t* ids, float* weights, void* lat, void* stream) {
  if (!fused || !bias || !ids || !weights || (latent > 0 && !lat)) return HB_ENULL;
  if (m <= 0 || e <= 0 || k <= 0 || k > e || k > 64 || e > 64 * ROUTE_PER_LANE || latent < 0 || stride < (int64_t)e + latent || steps <= 0)
    return HB_EINVAL;
  RouteParams p{};
  p.logits = fused;
  p.stride = stride;
  p.bias = bias;
  p.slots = slots;
  p.steps = steps;
  p.repeat = repeat;
  p.e = e;
  p.k = k;
  p.per = (e + 63) / 64;
  p.pad_id = e;
  p.latent = latent;
  p.ids = ids;
  p.weights = weights;
  p.lat = static_cast<uint16_t*>(lat);
  launch_route<true>(p, m, as_stream(stream));
  return launch_status();
}

static std::mutex g_trace_lock;
static int64_t* g_trace = nullptr;
static int64_t g_trace_records = 0;
int64_t* hb::moe_trace_buffer(int64_t* records) {
  std::lock_guard<std::mutex> hold(g_trace_lock);
  *records = g_trace_records;
  return g_trace;
}
#ifndef HB_NO_DEBUG_HOOKS
extern "C" int hb_debug_trace(void* buffer, int64_t records) {
  if (records < 0 || !aligned(buffer, 8)) return HB_EINVAL;
  std::lock_guard<std::mutex> hold(g_trace_lock);
  g_trace = records > 0 ? static_cast<int64_t*>(buffer) : nullptr;
  g_trace_records = g_trace ? records : 0;
  return HB_OK;
}

extern "C" int hb_debug_events(void* const* events, int count) {
  if (count < 0 || (count > 0 && !events)) return HB_EINVAL;
  std::lock_guard<std::mutex> hold(g_events_lock);
  g_events.assign(reinterpret_cast<hipEvent_t const*>(events), reinterpret_cast<hipEvent_t const*>(events) + count);
  g_event_next = 0;
  g_events_armed.store(count > 0, std::memory_order_relaxed);
  return HB_OK;
}
#endif

// Minor: what was added since 1.0 (the small latent block, hb_nvfp4_gemm_ws, budgeted routing, the layer under a budget, the
// ring skeleton hook, hb_workspace_reset / hb_workspace_status with the counters in the caller's workspace; 1.6: the layer from
// its rows, hb_nvfp4_gemm_room_bytes, the calls on a range of the experts, and other bytes in an NVFP4 tile layout).
extern "C" int hb_version(void) { return 1009; }

extern "C" const char* hb_error_string(int code) {
  switch (code) {
    case HB_OK: return "ok";
    case HB_EINVAL: return "unsupported shape, alignment or flag";
    case HB_ENULL: return "a required pointer is null";
    case HB_EWORKSPACE: return "workspace too small";
    case HB_ELAUNCH: return "the HIP runtime refused a launch";
    case HB_ESCRATCH: return "the call needs more scratch than the library's static buffer holds";
    default: return "unknown error";
  }
}
