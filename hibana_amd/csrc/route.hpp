// Top-k routing of one row by one wavefront (device code shared by the routing launches and by kernels that route for
// themselves).
#pragma once

#include "stream_common.hpp"

namespace hb {

// Top-k routing, one wavefront per row: softmax over all experts, top-k, renormalized
// (hibana/kernels/flashnext_fused.py:278-319 of the reference), or sigmoid scores chosen by score + bias with the plain
// scores as weights (hibana/model/nemotron/moe.py:57-121). Lane l holds experts l * per .. l * per + per - 1 in
// registers as order-preserving 32-bit keys; among equal scores the lowest lane, then the lowest register, wins - the lowest
// expert id (top_ranked).
constexpr int ROUTE_PER_LANE = 16;

__device__ __forceinline__ uint32_t wave_max_u32(uint32_t x) {
  x = max(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0xB1, 0xF, 0xF, false));   // lane ^ 1
  x = max(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x4E, 0xF, 0xF, false));   // lane ^ 2
  x = max(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x141, 0xF, 0xF, false));  // mirror within 8
  x = max(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x140, 0xF, 0xF, false));  // mirror within 16
  const uint32_t a = __builtin_amdgcn_readlane((int)x, 0), b = __builtin_amdgcn_readlane((int)x, 16);
  const uint32_t c = __builtin_amdgcn_readlane((int)x, 32), d = __builtin_amdgcn_readlane((int)x, 48);
  return max(max(a, b), max(c, d));
}

// The largest of a value over the wavefront (NaN only if all are), in every lane.
__device__ __forceinline__ float wave_max(float x) {
  x = fmaxf(x, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0xB1, 0xF, 0xF, false)));
  x = fmaxf(x, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x4E, 0xF, 0xF, false)));
  x = fmaxf(x, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x141, 0xF, 0xF, false)));
  x = fmaxf(x, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x140, 0xF, 0xF, false)));
  const int bits = __builtin_bit_cast(int, x);
  const float a = __builtin_bit_cast(float, __builtin_amdgcn_readlane(bits, 0)), b = __builtin_bit_cast(float, __builtin_amdgcn_readlane(bits, 16));
  const float c = __builtin_bit_cast(float, __builtin_amdgcn_readlane(bits, 32)), d = __builtin_bit_cast(float, __builtin_amdgcn_readlane(bits, 48));
  return fmaxf(fmaxf(a, b), fmaxf(c, d));
}

// Key of a score: larger score <=> larger key, every real key above 0 (the key of an empty register).
__device__ __forceinline__ uint32_t score_key(float v) {
  const int32_t bits = __builtin_bit_cast(int32_t, v);
  return (uint32_t)(bits ^ ((bits >> 31) & 0x7fffffff)) ^ 0x80000000u;
}

// Inclusive prefix sum over the wavefront's lanes without LDS: shifts within rows of sixteen lanes, then the rows' last
// lanes broadcast to the rows after them (DPP).
__device__ __forceinline__ int wave_inclusive_sum(int x) {
  x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xF, 0xF, false);  // row_shr:1
  x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xF, 0xF, false);  // row_shr:2
  x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xF, 0xF, false);  // row_shr:4
  x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xF, 0xF, false);  // row_shr:8
  x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xA, 0xF, false);  // row_bcast:15 into rows 1 and 3
  x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xC, 0xF, false);  // row_bcast:31 into rows 2 and 3
  return x;
}

// The k largest of a wavefront's keys (0: no key), largest first, one a lane: lane s < k gets selection s's key and its tag, the
// lane's place of it (lane * per + register). Equal keys in ascending lane, then register.
//
// A threshold that at least k lanes' largest keys reach, found by cutting the interval in four a step; where more than 63 keys
// reach it (rows of more than some 36 selections), raised until 63 or fewer do. Those go to a lane each (ds_permute), every lane
// counts the ones ahead of its own, and they go to the lanes their ranks name. TIES: equal keys are common (softmax scores of BF16
// logits: six rows in ten tie inside or at the end of the top 10 of 512), and the count goes by key and lane at once; else by the
// keys alone, and again where two lanes get one rank. What bounds it is one wavefront's chain of dependent instructions. The routing
// launch of 64 rows of 512 softmax scores, us, by rounds on sorted lists and so: top 10 4.7 and 4.1, top 22 6.3 and 4.9, top 40 8.8 and
// 6.2, top 56 11.0 and 7.1; scores of BF16 logits counted by the keys alone first, 4.7 and 6.0 at 10 and 22, so 4.1 and 4.9. One token of the three-bit
// layer (top 10 of 512) 19.8 us by rounds, 19.2 so; the latent block's one token (top 22) 47.4 and 46.0.
// Rounds, a selection each, remain for more than TOP_SEARCH selections, which leave the threshold too little room between k and 63
// keys (ties among 64 rows of BF16 logits: at 60 selections 14.4 us with the search in vain ahead of the rounds, 11.5 without), and for rows
// of many equal scores at it.
constexpr int TOP_SLACK = 3;    // lanes that may reach the threshold beyond k
constexpr int TOP_SEARCH = 56;  // selections, at most, that the threshold serves
template <bool TIES, int PER>
__device__ __forceinline__ void top_ranked(uint32_t (&key)[PER], int per, int k, int lane, uint32_t& out_key, int& out_tag) {
  out_key = 0u;
  out_tag = 0;
  if (__builtin_expect(k <= TOP_SEARCH, 1)) {  // uniform
    uint32_t head = key[0];
#pragma unroll
    for (int j = 1; j < PER; j++) head = max(head, key[j]);
    const uint32_t most = wave_max_u32(head), least = ~wave_max_u32(~head);
    uint32_t lo = max(least, 1u), hi = most;  // at least k lanes reach lo (or all that hold a key do); fewer than k reach hi, unless it is the threshold
    if (__popcll(__ballot(head >= hi)) >= k) lo = hi;
    while (hi - lo > 1u) {  // three places of the interval a step, their ballots side by side
      const uint32_t part = max((hi - lo) >> 2, 1u);
      const uint32_t at1 = lo + part, at2 = min(at1, hi - part) + part, at3 = min(at2, hi - part) + part;
      const int reach1 = __popcll(__ballot(head >= at1)), reach2 = __popcll(__ballot(head >= at2)), reach3 = __popcll(__ballot(head >= at3));
      const bool over1 = reach1 >= k, over2 = reach2 >= k, over3 = reach3 >= k;
      const int reach = over3 ? reach3 : over2 ? reach2 : over1 ? reach1 : 64;
      hi = over3 ? hi : over2 ? at3 : over1 ? at2 : at1;
      lo = over3 ? at3 : over2 ? at2 : over1 ? at1 : lo;
      if (reach <= k + TOP_SLACK) break;
    }
    auto reaching = [&] {
      int n = 0;
#pragma unroll
      for (int j = 0; j < PER; j++) n += key[j] >= lo ? 1 : 0;
      return n;
    };
    int count = reaching(), upto = wave_inclusive_sum(count), all = __builtin_amdgcn_readlane(upto, 63);
    if (__builtin_expect(all > 63, 0)) {  // uniform
      uint32_t over = most;
      while (over - lo > 1u && all > 63) {
        const uint32_t mid = lo + ((over - lo) >> 1);
        int n = 0;
#pragma unroll
        for (int j = 0; j < PER; j++) n += __popcll(__ballot(key[j] >= mid));
        if (n >= k) lo = mid, all = n; else over = mid;
      }
      count = reaching();
      upto = wave_inclusive_sum(count);
    }
    if (__builtin_expect(all <= 63, 1)) {  // (all >= k, or every key there is)
      int at = upto - count;
      uint32_t mine = 0u;
      int tag = 0;
#pragma unroll
      for (int j = 0; j < PER; j++) {  // lane 63 takes what goes nowhere; a lane that nothing is sent to gets zero
        const bool take = key[j] >= lo;
        const int to = 4 * (take ? at : 63);
        mine |= (uint32_t)__builtin_amdgcn_ds_permute(to, (int)key[j]);
        tag |= __builtin_amdgcn_ds_permute(to, lane * per + j);
        at += take ? 1 : 0;
      }
      if (lane >= all) mine = 0u;
      const uint32_t under = mine - 1u;  // a lower lane's equal key is ahead: it exceeds the key less one (no key here is 0)
      auto deal = [&](bool ties) {
        int rank = 0;
        for (int c0 = 0; c0 < all; c0 += 4) {
#pragma unroll
          for (int c = 0; c < 4; c++) {
            const uint32_t other = (uint32_t)__builtin_amdgcn_readlane((int)mine, min(c0 + c, 63));
            rank += other > (ties && __builtin_amdgcn_inverse_ballot_w64(~1ull << min(c0 + c, 63)) ? under : mine) ? 1 : 0;
          }
        }
        const int to = 4 * (lane < all && rank < k ? rank : 63);
        out_key = (uint32_t)__builtin_amdgcn_ds_permute(to, (int)mine);
        out_tag = __builtin_amdgcn_ds_permute(to, tag);
        return TIES || __popcll(__ballot(lane < all && rank < k)) == __popcll(__ballot(lane < k && out_key != 0u));  // a rank for every key, a key for every rank
      };
      if (__builtin_expect(!deal(TIES), 0)) deal(true);  // equal keys had one rank between them
      if (lane >= k) out_key = 0u, out_tag = 0;
      return;
    }
  }
  // The lane's keys in descending order once (adjacent exchanges on a strictly larger right neighbour only, so equal keys keep
  // their order), their registers as nibbles of one word: a round looks at the heads, and the winner's list moves up by one.
  uint32_t from[PER];
#pragma unroll
  for (int j = 0; j < PER; j++) from[j] = j;
#pragma unroll
  for (int pass = 0; pass < PER; pass++) {
#pragma unroll
    for (int j = pass & 1; j + 1 < PER; j += 2) {
      const bool swap = key[j + 1] > key[j];
      const uint32_t ka = key[j], kb = key[j + 1], fa = from[j], fb = from[j + 1];
      key[j] = swap ? kb : ka;
      key[j + 1] = swap ? ka : kb;
      from[j] = swap ? fb : fa;
      from[j + 1] = swap ? fa : fb;
    }
  }
  uint64_t order = 0;
#pragma unroll
  for (int j = 0; j < PER; j++) order |= (uint64_t)from[j] << (4 * j);
  for (int s = 0; s < k; s++) {
    const uint32_t top = wave_max_u32(key[0]);
    const int winner = __builtin_ctzll(__ballot(key[0] == top));
    const int from_register = __builtin_amdgcn_readlane((int)order, winner) & 15;
    if (lane == s) {
      out_key = top;
      out_tag = winner * per + from_register;
    }
    if (lane == winner) {
#pragma unroll
      for (int j = 0; j + 1 < PER; j++) key[j] = key[j + 1];
      key[PER - 1] = 0u;
      order >>= 4;
    }
  }
}

struct RouteParams {
  const float* logits;   // [m, stride]: e logits a row (sigmoid: followed by `latent` FP32 columns)
  int64_t stride;
  const float* bias;     // sigmoid: [e] added to the scores for the choice only
  const int32_t* slots;  // row r is real iff slots[r / steps] != 0 (null: every row)
  int steps, repeat;
  int e, k, per, latent;
  int pad_id;            // the id of a padded row's slots without `repeat` (the callers' default: e, "no expert")
  int sigmoid;           // the rule a kernel that serves both applies (route_any)
  int half;              // softmax: `logits` points to BF16 values (read as FP32: the router's product as it was rounded)
  int32_t* ids;
  float* weights;
  uint16_t* lat;         // sigmoid: BF16 [m, latent], the row's latent columns
  float* raw;            // or null: [m, k], the weights before renormalization (a padded row: those of the row it repeats)
};

// THROUGH: the logits were written by other workgroups of the same launch and are read past the compute die's L2.
// Returns, in lane s < k, the id of the row's selection s. `write` = false keeps the row's results in registers only (a
// workgroup that routes for itself a row some other workgroup writes).
template <bool SIGMOID, int PER, bool THROUGH = false>
__device__ __forceinline__ int route_row(const RouteParams& p, int r, int lane, bool write = true, float* weight = nullptr) {
  const int e = p.e, per = p.per, first = lane * per;
  auto logit = [](const float* at) -> float { if constexpr (THROUGH) return load_through(at); else return *at; };
  const bool padded = p.slots && p.slots[r / p.steps] == 0;  // asked for first: the answer picks the row the logits are read from
  if (SIGMOID && p.lat && write) {  // the row's latent columns, rounded: four a lane and sixteen loads in flight where the row allows
    const float* src = p.logits + (int64_t)r * p.stride + e;
    uint16_t* dst = p.lat + (int64_t)r * p.latent;
    if (!THROUGH && !((p.stride | e | p.latent) & 3)) {
      for (int c0 = 4 * lane; c0 < p.latent; c0 += 1024) {
        f32x4_t v[4];
#pragma unroll
        for (int j = 0; j < 4; j++)
          if (c0 + 256 * j < p.latent) v[j] = *reinterpret_cast<const f32x4_t*>(src + c0 + 256 * j);
#pragma unroll
        for (int j = 0; j < 4; j++)
          if (c0 + 256 * j < p.latent) {
            const uint32_t lo = (uint32_t)bf16_of(v[j].x) | ((uint32_t)bf16_of(v[j].y) << 16), hi = (uint32_t)bf16_of(v[j].z) | ((uint32_t)bf16_of(v[j].w) << 16);
            *reinterpret_cast<uint2*>(dst + c0 + 256 * j) = make_uint2(lo, hi);
          }
      }
    } else {
      for (int c = lane; c < p.latent; c += 64) dst[c] = bf16_of(logit(src + c));
    }
  }
  const float* row = p.logits + (int64_t)(padded ? 0 : r) * p.stride;  // a padded row repeats row 0's first choice
  const uint16_t* row16 = reinterpret_cast<const uint16_t*>(p.logits) + (int64_t)(padded ? 0 : r) * p.stride;
  float val[PER];   // the weight an expert would get before renormalization
  uint32_t key[PER];
  float lg[PER];    // the lane's logits: every load is asked for before the first is used
  if (!THROUGH && PER == 8 && per == 8 && e == 512 && !p.half && !((p.stride | (int64_t)(reinterpret_cast<uintptr_t>(p.logits) >> 2)) & 3)) {
    // the lane's eight logits are 32 consecutive bytes on a 16-byte boundary: two loads instead of eight
    const f32x4_t lo = *reinterpret_cast<const f32x4_t*>(row + first), hi = *reinterpret_cast<const f32x4_t*>(row + first + 4);
    lg[0] = lo.x, lg[1] = lo.y, lg[2] = lo.z, lg[3] = lo.w;
    if constexpr (PER >= 8) lg[4] = hi.x, lg[5] = hi.y, lg[6] = hi.z, lg[7] = hi.w;
  } else if (!SIGMOID && p.half) {
    if (PER == 8 && per == 8 && e == 512 && !(reinterpret_cast<uintptr_t>(row16) & 15)) {  // ... and one for eight BF16
      const u32x4_t v = *reinterpret_cast<const u32x4_t*>(row16 + first);
#pragma unroll
      for (int j = 0; j < 4; j++) {
        lg[2 * j] = __uint_as_float(v[j] << 16);
        lg[2 * j + 1] = __uint_as_float(v[j] & 0xffff0000u);
      }
    } else {
#pragma unroll
      for (int j = 0; j < PER; j++) lg[j] = bf16_bits_to_f32(row16[min(first + j, e - 1)]);
    }
  } else {
#pragma unroll
    for (int j = 0; j < PER; j++) lg[j] = logit(row + min(first + j, e - 1));
  }
  if (SIGMOID) {
    float bs[PER];
#pragma unroll
    for (int j = 0; j < PER; j++) bs[j] = p.bias[min(first + j, e - 1)];
#pragma unroll
    for (int j = 0; j < PER; j++) {
      const bool real = j < per && first + j < e;
      val[j] = real ? 1.0f / (1.0f + expf(-lg[j])) : 0.f;
      key[j] = real ? score_key(val[j] + bs[j]) : 0u;
    }
  } else {
    float mx = -INFINITY;
#pragma unroll
    for (int j = 0; j < PER; j++) {
      val[j] = j < per && first + j < e ? lg[j] : -INFINITY;
      mx = fmaxf(mx, val[j]);
    }
    mx = wave_max(mx);
    float sum = 0.f;
#pragma unroll
    for (int j = 0; j < PER; j++) {
      val[j] = j < per && first + j < e ? expf(val[j] - mx) : 0.f;
      sum += val[j];
    }
    sum = wave_sum(sum);
#pragma unroll
    for (int j = 0; j < PER; j++) {
      val[j] = val[j] / sum;
      key[j] = j < per && first + j < e ? score_key(val[j]) : 0u;
    }
  }
  float total = 0.f, mine = 0.f;
  int mine_id;
  uint32_t mine_key;
  top_ranked<!SIGMOID>(key, per, p.k, lane, mine_key, mine_id);
  if (lane < p.k) {
    if (SIGMOID) {  // the key is score + bias: the plain score is made again from the logit
      mine = 1.0f / (1.0f + expf(-logit(row + mine_id)));
    } else {        // the key is the probability's own bits
      const uint32_t u = mine_key ^ 0x80000000u;
      mine = __builtin_bit_cast(float, u ^ (uint32_t)(((int32_t)u >> 31) & 0x7fffffff));
    }
  }
  for (int s = 0; s < p.k; s++) total += __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, mine), s));  // in rank order
  int id = mine_id;
  float w = SIGMOID ? mine / (total + 1e-20f) : mine / total;
  if (padded) {
    id = p.repeat ? __builtin_amdgcn_readfirstlane(mine_id) : p.pad_id;
    w = 0.f;
  }
  if (lane < p.k && write) {
    store_through(&p.ids[(int64_t)r * p.k + lane], id);  // the plan may read it in this very launch, from another workgroup
    p.weights[(int64_t)r * p.k + lane] = w;
    if (p.raw) p.raw[(int64_t)r * p.k + lane] = mine;
  }
  if (weight) *weight = w;
  return id;
}

// Row r by the rule and the register count the parameters name.
__device__ __forceinline__ void route_any(const RouteParams& p, int r, int lane) {
  if (p.sigmoid) {
    if (p.per <= 8) {
      route_row<true, 8>(p, r, lane);
    } else {
      route_row<true, 16>(p, r, lane);
    }
  } else if (p.per <= 8) {
    route_row<false, 8>(p, r, lane);
  } else {
    route_row<false, 16>(p, r, lane);
  }
}

}  // namespace hb
