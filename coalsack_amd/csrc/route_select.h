// Per-token expert selection (top-k, close calls recomputed in the reference's summation
// order, routing weights) and the dispatch of a small batch, as device functions of the
// router kernels.
#pragma once
#include "common.h"

namespace csk {

// --------------------------------------------------- per-token selection
// Maximum over the 64 lanes, the same value returned in every lane: four cross-lane steps
// inside each row of 16 (quad swaps, half-row and row mirrors: ordinary vector-ALU latency,
// where a shuffle through the LDS crossbar takes ten times as long) and the four row
// results combined through scalar registers.
template <int CTRL>
__device__ __forceinline__ float dpp_max(float a) {
  const int x = __float_as_int(a);
  return fmaxf(a, __int_as_float(__builtin_amdgcn_update_dpp(x, x, CTRL, 0xf, 0xf, false)));
}
__device__ __forceinline__ float wave_max_all(float v) {
  v = dpp_max<0xB1>(v);   // quad_perm [1,0,3,2]
  v = dpp_max<0x4E>(v);   // quad_perm [2,3,0,1]
  v = dpp_max<0x141>(v);  // row_half_mirror
  v = dpp_max<0x140>(v);  // row_mirror
  const int x = __float_as_int(v);
  const float r0 = __int_as_float(__builtin_amdgcn_readlane(x, 0));
  const float r1 = __int_as_float(__builtin_amdgcn_readlane(x, 16));
  const float r2 = __int_as_float(__builtin_amdgcn_readlane(x, 32));
  const float r3 = __int_as_float(__builtin_amdgcn_readlane(x, 48));
  return fmaxf(fmaxf(r0, r1), fmaxf(r2, r3));
}

// Lanes 0..k hold the k+1 largest logits in descending order (fewer when E == k): the lanes whose logit and the next one are
// closer than tol.
__device__ __forceinline__ unsigned long long close_pairs(float my_val, int lane, int E, int k, float tol) {
  // the value one lane up (wave_shl:1, a vector-ALU operation): no trip through the LDS crossbar
  const int mv = __float_as_int(my_val);
  const float below = __int_as_float(__builtin_amdgcn_update_dpp(mv, mv, 0x130, 0xf, 0xf, false));
  return __ballot(lane < k && lane + 1 < E && (my_val - below) <= tol * fmaxf(1.0f, fabsf(my_val)));
}

// The logits that a close call puts in question are those in [lo, hi]: from the first member of a close pair to the last; where the
// last pair's lower member is the runner-up, a safe margin below it too, since what is there might outrank it.  All others
// keep their tree-ordered values, which differ from their neighbours' by more than both can move.  (A function of its own, for the
// callers that have a close call: inside select_topk it took 0.4 us of the one-token kernel, which then held more values than
// it has scalar registers.)
__device__ __forceinline__ void close_call_range(float my_val, int lane, int E, int k, float tol, float& lo, float& hi) {
  const unsigned long long pairs = close_pairs(my_val, lane, E, k, tol);  // not empty
  const int mv = __float_as_int(my_val);
  const int first = (int)__builtin_ctzll(pairs), last = 64 - (int)__builtin_clzll(pairs);
  hi = __int_as_float(__builtin_amdgcn_readlane(mv, first));
  lo = __int_as_float(__builtin_amdgcn_readlane(mv, last));
  if (last == k) lo = lo - 2.0f * tol * fmaxf(1.0f, fabsf(lo));
  asm volatile("" : "+v"(lo), "+v"(hi));  // kept in vector registers: the one-token kernel has no scalar ones to spare
}

// One wave selects one token's top k.  Lane l holds the logits of experts l, l+64,
// l+128, l+192; each round finds the wave-wide maximum, locates its owner with ballots
// (ties -> lowest expert index) and retires it.  One round more than k records
// the runner-up, so that the k+1 largest logits are known: if any two adjacent ones are
// closer than the difference between this library's tree-ordered fp32 sums and the
// reference's strictly sequential ones can be (moe_router_node.h:161-167: sum += h*g,
// multiply and add rounded separately, bias added last), the caller recomputes the
// logits in question in exactly that order and selects again -- so the expert indices
// and their slot order equal the reference's whenever the inputs are the same, not only
// when no two logits are close.  Lane s < k returns slot s in (my_val, my_idx).
//
// The k experts returned are always distinct and below E, whatever the logits hold -- the
// dispatch and the one-token launch (k token groups, known before the kernel runs) rely on
// it.  Retired and out-of-range entries are -inf; the logits compete as max(logit, -FLT_MAX),
// which turns a NaN or a -inf into the lowest finite key, so that such a logit is still a
// candidate distinct from the retired ones (among equal keys the lowest index wins).  A token
// whose logits hold a NaN or +inf, or nothing but -inf, has NaN routing weights in the
// reference's softmax (moe_router_node.h:176-200: exp(inf - inf), or a NaN sum); which experts
// its partial sort then returns is unspecified.  Here such a token gets NaN in every slot's value, hence NaN
// weights, k distinct experts, and no close-call recomputation.
__device__ __forceinline__ void select_topk(float (&v)[4], int lane, int E, int k, float& my_val,
                                            int& my_idx, float& vmax, bool& close_call, float tol) {
  const float NEG = -__builtin_inff();
  constexpr float kLowest = -3.402823466e+38f;
  bool bad = false, finite = false;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const bool real = lane + 64 * j < E;
    bad = bad || (real && !(v[j] <= -kLowest));           // NaN or +inf
    finite = finite || (real && fabsf(v[j]) <= -kLowest);
    if (real) v[j] = fmaxf(v[j], kLowest);
  }
  const bool poisoned = __any(bad) || !__any(finite);      // (every logit -inf: exp(-inf + inf))
  my_val = 0.0f, my_idx = 0, vmax = 0.0f;
  for (int s = 0; s <= k; ++s) {
    const float best = wave_max_all(fmaxf(fmaxf(v[0], v[1]), fmaxf(v[2], v[3])));
    // its owner: lowest expert index among equals = lowest register j, then lowest lane
    int bi = 0;
    bool found = false;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const unsigned long long m = __ballot(v[j] == best);
      if (!found && m != 0ull) {
        bi = (int)__builtin_ctzll(m) + 64 * j;
        found = true;
      }
    }
    if (s == 0) vmax = best;
    if (lane == s) {
      my_val = best;
      my_idx = bi;
    }
    if (s < k && (bi & 63) == lane) {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if ((bi >> 6) == j) v[j] = NEG;
    }
  }
  close_call = close_pairs(my_val, lane, E, k, tol) != 0ull && !poisoned;
  if (poisoned) {
    my_val = __builtin_nanf("");
    vmax = my_val;
  }
}

// Logits in the reference's order: a strictly sequential fp32 sum per logit, multiply and
// add rounded separately (moe_router_node.h:161-167).  The chain of H dependent additions
// cannot be reordered, but everything else can be taken out of its way: the whole workgroup
// multiplies (coalesced loads, the products do not depend on the running sum) and stages
// the rounded products in LDS, the waves then only read back and add.
//
// A few logits (as a rule two: a close pair): the chain is cut into segments that run side by side, a wave each.  A segment
// needs the exact sum in front of it, which is not known yet -- but it is known to a few units in the last place, from a sum in
// any order, and a wave has 64 lanes: each lane adds the segment's products to a sum of its own, the approximate one and
// the 63 floating-point numbers around it.  When the segment before is done its end is looked up among them, bit for
// bit, and the segment's end is that lane's.  Where no lane began there (7 to 12 % of the segments of 2880 normally
// distributed products in four) the segment is added again from its true beginning.  The result is the chain's either way.
// Many logits: a row per lane of wave 0, all rows side by side, products one chunk of K ahead.
// A dependent addition takes 8 cycles, 2880 of them 15 us at the 1.5 GHz that a long prompt's GEMMs leave the part at.  The launch
// with a close call in it: 2048 tokens on 32 experts 31.0 -> 21 us, 4096 on 128 38 -> 27 (8 waves, two rows in four segments);
// 50 tokens of eight layers, top-8, whose nine largest logits were recomputed in two rounds whichever were close, 515 -> 506 us
// on average over inputs.
constexpr int kCcBatch = 8;              // logits recomputed side by side
constexpr int kCcChunk = 768;            // elements of K staged per step
constexpr int kCcSplitFloats = 6144;     // products staged at once where chains are cut

template <int NT, int B, int CH = kCcChunk>
struct CloseCallLdsT {
  static constexpr int kCcStride = CH + 4;  // LDS row stride: rows start four banks apart
  alignas(16) float prod[2][B][kCcStride];
  static constexpr bool kCut = CH == kCcChunk;  // (the smaller area is that of the one-token kernel, which has none to spare)
  static_assert(!kCut || 2 * B * kCcStride >= kCcSplitFloats + 64, "reads run up to 64 products past the last row's end");
  float ends[kCut ? NT / 64 : 1][kCut ? 64 : 1];  // per segment: the lanes' sums ...
  int around[kCut ? NT / 64 : 1];                 // ... and the bits of the number that lane 32 began with
  float carry[B];                                 // per row: the sum so far
  float fixed[kMaxExperts];  // the token's logits, recomputed ones replaced
  int cand[kMaxExperts];
  int ncand;
};

// sum + the products of n4 (a multiple of 8) quads in LDS, one after the other, in every lane; quads up to 4 past them are read
__device__ __forceinline__ float add_in_order(const floatx4* q, int n4, float sum) {
#pragma clang fp contract(off)
  floatx4 qa[4], qb[4];
  auto rd = [&](floatx4(&r)[4], int i0) {
#pragma unroll
    for (int i = 0; i < 4; ++i) r[i] = q[i0 + i];
  };
  auto add = [&](const floatx4(&r)[4]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      sum = sum + r[i][0];
      sum = sum + r[i][1];
      sum = sum + r[i][2];
      sum = sum + r[i][3];
    }
  };
  rd(qa, 0);
  for (int i0 = 0; i0 < n4; i0 += 8) {
    rd(qb, i0 + 4);
    add(qa);
    rd(qa, i0 + 8);
    add(qb);
  }
  return sum;
}

// The m logits of s.cand (at least two, at most NT / 128 and kCcBatch), chains cut into segments.
template <int NT, int B, int CH>
__device__ __forceinline__ void logits_reference_order_cut(const float* __restrict__ x, const float* __restrict__ g,
                                                           const float* __restrict__ b, int H4, int m,
                                                           CloseCallLdsT<NT, B, CH>& s) {
#pragma clang fp contract(off)
  constexpr int NW = NT / 64, kQuads = kCcSplitFloats / 4;
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const CSK_GLOBAL floatx4* x4 = as_global(reinterpret_cast<const floatx4*>(x));
  const CSK_GLOBAL floatx4* g4 = as_global(reinterpret_cast<const floatx4*>(g));
  const int R = m <= 2 ? 2 : m <= 4 ? 4 : 8, S = NW / R;  // rows, segments of a row: powers of two
  const int row4 = kQuads / R;                            // quads of a row that are staged at once
  const int nb = (H4 + row4 - 1) / row4, per = (H4 + nb - 1) / nb;
  const int seg4 = ((per + S - 1) / S + 7) & ~7;          // S * seg4 <= row4: row4 / S is a multiple of 8
  floatx4* const prod = reinterpret_cast<floatx4*>(&s.prod[0][0][0]);
  const int c = wv / S, j = wv - c * S;
  const floatx4* const row = prod + c * row4;
  float sum = 0.0f;
  for (int h0 = 0; h0 < H4; h0 += per) {
    const int n4 = min(per, H4 - h0);
    constexpr int kItems = (kQuads + NT - 1) / NT;
    floatx4 xq[kItems], gq[kItems];
#pragma unroll
    for (int it = 0; it < kItems; ++it) {
      const int idx = tid + it * NT, r = idx * R / kQuads, i4 = idx - r * row4;
      xq[it] = gq[it] = floatx4{0.f, 0.f, 0.f, 0.f};  // behind the row's end: adding a zero changes no sum
      if (r < m && i4 < n4) {
        xq[it] = x4[h0 + i4];
        gq[it] = g4[(size_t)s.cand[r] * H4 + h0 + i4];
      }
    }
#pragma unroll
    for (int it = 0; it < kItems; ++it)
      if (tid + it * NT < kQuads) prod[tid + it * NT] = xq[it] * gq[it];
    __syncthreads();
    if (c < m) {
      if (j > 0) {
        float a = 0.0f;
        for (int i = lane; i < j * seg4; i += 64) a += (row[i][0] + row[i][1]) + (row[i][2] + row[i][3]);
        const int around = __float_as_int(sum + wave_sum(a));
        const float end = add_in_order(row + j * seg4, seg4, __int_as_float(around + lane - 32));
        s.ends[wv][lane] = end;
        if (lane == 0) s.around[wv] = around;
      } else {
        sum = add_in_order(row, seg4, sum);
      }
    }
    __syncthreads();
    if (c < m && j == 0) {
      for (int i = 1; i < S; ++i) {
        const unsigned at = (unsigned)(__float_as_int(sum) - s.around[wv + i] + 32);
        sum = at < 64u ? s.ends[wv + i][at] : add_in_order(row + i * seg4, seg4, sum);
      }
      s.carry[c] = sum;
    }
    __syncthreads();
    if (c < m) sum = s.carry[c];
  }
  if (c < m && j == 0 && lane == 0) {
    const int e = s.cand[c];
    s.fixed[e] = sum + (b ? b[e] : 0.0f);
  }
  __syncthreads();
}

// Called by all NT threads of the workgroup with the same arguments.  Recomputes the
// logits in [lo, hi] (select_topk) and leaves all E logits of the
// token in s.fixed.  H must be a multiple of 4.
template <int NT, int B, int CH>
__device__ __forceinline__ void logits_reference_order_wg(const float* __restrict__ x,
                                                          const float* __restrict__ g,
                                                          const float* __restrict__ b,
                                                          const float* __restrict__ logit_row, int E,
                                                          int H, float lo, float hi, CloseCallLdsT<NT, B, CH>& s) {
#pragma clang fp contract(off)
  constexpr int kC4 = CH / 4;
  constexpr int kProducers = NT - 64;  // wave 0 only adds
  constexpr int kItems = (B * kC4 + kProducers - 1) / kProducers;
  const int tid = threadIdx.x, ptid = tid - 64;
  if (tid == 0) s.ncand = 0;
  __syncthreads();
  for (int e = tid; e < E; e += NT) {
    const float v = logit_row[e];
    s.fixed[e] = v;
    if (v >= lo && v <= hi) s.cand[atomicAdd(&s.ncand, 1)] = e;
  }
  __syncthreads();
  const int m = s.ncand;
  const CSK_GLOBAL floatx4* x4 = as_global(reinterpret_cast<const floatx4*>(x));
  const CSK_GLOBAL floatx4* g4 = as_global(reinterpret_cast<const floatx4*>(g));
  const int H4 = H >> 2;
  if constexpr (CloseCallLdsT<NT, B, CH>::kCut) {
    if (m <= min(NT / 128, B)) {
      logits_reference_order_cut<NT>(x, g, b, H4, m, s);
      return;
    }
  }
  const int nchunk = (H4 + kC4 - 1) / kC4;
  for (int c0 = 0; c0 < m; c0 += B) {
    const int mb = min(B, m - c0);
    // producers: rounded products of chunk ci of the batch's rows -> LDS buffer ci & 1
    auto produce = [&](int ci) {
      const int h4 = ci * kC4, len4 = min(kC4, H4 - h4);
      floatx4 xq[kItems], gq[kItems];
#pragma unroll
      for (int it = 0; it < kItems; ++it) {
        const int idx = ptid + it * kProducers, c = idx / kC4, i4 = idx - c * kC4;
        if (c < mb) {
          const int i = h4 + min(i4, len4 - 1);
          xq[it] = x4[i];
          gq[it] = g4[(size_t)s.cand[c0 + c] * H4 + i];
        }
      }
#pragma unroll
      for (int it = 0; it < kItems; ++it) {
        const int idx = ptid + it * kProducers, c = idx / kC4, i4 = idx - c * kC4;
        const floatx4 p = xq[it] * gq[it];
        // behind the row's end: adding a zero changes no sum
        if (c < mb) *reinterpret_cast<floatx4*>(&s.prod[ci & 1][c][4 * i4]) = i4 < len4 ? p : floatx4{0.f, 0.f, 0.f, 0.f};
      }
    };
    if (ptid >= 0) produce(0);
    __syncthreads();
    float sum = 0.0f;
    for (int ci = 0; ci < nchunk; ++ci) {
      if (ptid >= 0) {
        if (ci + 1 < nchunk) produce(ci + 1);  // while wave 0 adds chunk ci
      } else if (tid < mb) {
        const int len4 = min(kC4, H4 - ci * kC4);
        // (reads run into the next row or what lies behind the last one: never added)
        sum = add_in_order(reinterpret_cast<const floatx4*>(&s.prod[ci & 1][tid][0]), (len4 + 7) & ~7, sum);
      }
      __syncthreads();
    }
    if (tid < mb) {
      const int e = s.cand[c0 + tid];
      s.fixed[e] = sum + (b ? b[e] : 0.0f);
    }
    __syncthreads();
  }
}

// How close is a close call.  Measured over 1.3 million logits (six shapes, H from 256 to
// 2880): |tree-ordered sum - sequential sum| / max(1, |logit|) has an rms of 0.28 and a
// maximum of 2.3 in units of 2^-24 * sqrt(H) (the random-walk size of the sequential
// sum's rounding error); the tests hold the maximum below 3.  Two logits can change rank
// only if they are closer than the sum of their two differences; the threshold is 8 units,
// twice the largest pair of differences seen.  At gpt-oss shapes about one token in 2500
// is recomputed.
__device__ __forceinline__ float close_call_tolerance(int H) { return 8.0f * 5.96e-8f * sqrtf((float)H); }

// Routing weight of slot `lane` (moe_router_node.h:180-202): sigmoid of the raw logit, or
// softmax over the selected k with max subtraction, sum in slot order, multiply by 1/sum.
__device__ __forceinline__ float routing_weight(float my_val, float vmax, int lane, int k, int sigmoid) {
  if (sigmoid) return 1.0f / (1.0f + expf(-my_val));
  float w = (lane < k) ? expf(my_val - vmax) : 0.0f;
  float sum = 0.0f;
  for (int s = 0; s < k; ++s) sum += __int_as_float(__builtin_amdgcn_readlane(__float_as_int(w), s));  // slot order
  const float inv = (sum > 0.0f) ? (1.0f / sum) : 0.0f;
  return w * inv;
}

// Work descriptor of one active-expert slot (all zero when the slot is unused), written
// field by field: a local copy of the structure would live in scratch memory.
__device__ __forceinline__ void write_work_desc(WorkDesc* d, bool on, int e, int Te, int base,
                                                const ExpertW& w) {
  d->e = e;
  d->Te = on ? Te : 0;
  d->base = on ? base : 0;
  d->pad = 0;
  d->w.q_gate = on ? w.q_gate : nullptr;
  d->w.s_gate = on ? w.s_gate : nullptr;
  d->w.q_up = on ? w.q_up : nullptr;
  d->w.s_up = on ? w.s_up : nullptr;
  d->w.q_down = on ? w.q_down : nullptr;
  d->w.s_down = on ? w.s_down : nullptr;
  d->w.b_gate = on ? w.b_gate : nullptr;
  d->w.b_up = on ? w.b_up : nullptr;
  d->w.b_down = on ? w.b_down : nullptr;
}


constexpr int kRouteTinyTokens = 4;  // a wave of a workgroup of four selects for each
constexpr int kRouteTinyMaxP = 64;   // their assignments: one per lane
constexpr int kRouteFewTokens = 8;   // tokens that the gate/up kernel may route itself

// ------------------------------------- small batches: top-k + dispatch, fused
// One workgroup does, for P = T * k <= MAXP assignments, what router_topk_kernel and
// dispatch_scatter_kernel do in two launches: top-k and weights per token (one wave per
// token), per-expert counts, exclusive scan, ordered lists, and token groups or work descriptors and M
// tiles -- all through LDS.  A chain of dependent steps on one compute unit: none of them walks the experts or the list entries one
// after the other (ranks found by a ballot per distinct expert, four experts' groups written by one lane, and descriptors that
// nobody read, 16 tokens on 128 experts took 10.0 us; now 8.1, and the dispatch kernel of 50 tokens, which found its ranks
// the same way, 7.0 / 5.0; 8 layers of 64 experts of 2048 x 768, top-8, 50 tokens 528 -> 505 us).
constexpr int kListGroups = 0, kListDesc = 1;
struct RouteIn {
  const float* logits;  // [T, E]
  const float* x;       // [T, H] rows the logits were computed from (close calls are recomputed)
  const float* g;       // [E, H]
  const float* b;       // [E] or null
  const ExpertW* ew;    // [E]
  int T, E, k, H, sigmoid, group_tokens;
  int lists;  // what the expert kernels walk: kListGroups, or kListDesc (work descriptors and M tiles)
};
struct RouteOut {
  float* pairs;       // [T, k, 2]
  int* ids;           // [T * k]
  int* pos_of_slot;   // [T * k]
  int* counts;        // [E]
  int* offsets;       // [E + 1]
  WorkDesc* desc;     // [E]
  StreamGroup* groups;  // [token groups]
  int* nv;
  int* mtiles;        // [2 * M tiles]
  int* n_mtiles;
  int* list_tok;      // [T * k]
  float* list_w;      // [T * k]
};
// Inclusive prefix sum over the 64 lanes: shifts inside each row of 16 on the vector ALU
// (lanes without a source add zero), then the totals of the rows before through scalar
// registers.
template <int CTRL>
__device__ __forceinline__ int dpp_shr_add(int v) {
  return v + __builtin_amdgcn_update_dpp(0, v, CTRL, 0xf, 0xf, true);
}
__device__ __forceinline__ int wave_scan_inclusive(int v, int lane) {
  v = dpp_shr_add<0x111>(v);  // row_shr:1
  v = dpp_shr_add<0x112>(v);  // row_shr:2
  v = dpp_shr_add<0x114>(v);  // row_shr:4
  v = dpp_shr_add<0x118>(v);  // row_shr:8
  const int t0 = __builtin_amdgcn_readlane(v, 15), t1 = __builtin_amdgcn_readlane(v, 31);
  const int t2 = __builtin_amdgcn_readlane(v, 47);
  const int row = lane >> 4;
  return v + (row >= 1 ? t0 : 0) + (row >= 2 ? t1 : 0) + (row >= 3 ? t2 : 0);
}

// ceil(c / g) for the group sizes in use (64, 4 and 1) without a run-time integer division
__device__ __forceinline__ int group_count(int c, int g) { return g == 64 ? (c + 63) >> 6 : g == 4 ? (c + 3) >> 2 : c; }

template <int NT, int CCB, int MAXP>
struct RouteLds {
  int ids[MAXP];       // expert of assignment p = t * k + slot
  float wts[MAXP];     // its routing weight
  int cnt[kMaxExperts], off[kMaxExperts], act_e[kMaxExperts];
  int first[kMaxExperts], slot[kMaxExperts];  // the expert's first list entry (token group or M tile), its place among the active ones
  int na;
  unsigned long long named[MAXP / 64][kMaxExperts];  // per 64-assignment chunk: the assignments that name the expert
  short before[MAXP / 64][kMaxExperts];              // how many in the chunks before
  unsigned long long ew[kMaxExperts * (sizeof(ExpertW) / 8)];  // the experts' weight pointers, staged early
  CloseCallLdsT<NT, CCB> cc;
  int cc_tok[64], cc_n;
  float cc_lo[64], cc_hi[64];
};

template <int NT, int CCB, int MAXP>
__device__ __forceinline__ void route_workgroup(const RouteIn& r, const RouteOut& o, RouteLds<NT, CCB, MAXP>& s) {
  constexpr int NW = NT / 64;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int T = r.T, E = r.E, k = r.k;
  const int P = T * k;
  const float NEG = -__builtin_inff();
  const float tol = close_call_tolerance(r.H);
  static_assert(MAXP <= NT && MAXP % 64 == 0, "assignment p belongs to thread p, chunk p / 64 to wave p / 64");
  const int nchunk = (P + 63) >> 6;
  for (int i = threadIdx.x; i < nchunk * kMaxExperts; i += NT) (&s.named[0][0])[i] = 0ull;
  if (threadIdx.x == 0) s.cc_n = 0;
  // the table of weight pointers is needed last (work descriptors); its load is started
  // first, so that its latency runs beside that of the logits
  static_assert(sizeof(ExpertW) % 8 == 0, "copied as 64-bit words");
  static_assert(MAXP < 32768, "counts are scanned as 16-bit halves");
  constexpr int kEwWords = kMaxExperts * (int)(sizeof(ExpertW) / 8), kEwPerThread = (kEwWords + NT - 1) / NT;
  unsigned long long ew_reg[kEwPerThread];
#pragma unroll
  for (int i = 0; i < kEwPerThread; ++i) {
    const int w = threadIdx.x + i * NT;
    ew_reg[i] = w < E * (int)(sizeof(ExpertW) / 8) ? reinterpret_cast<const unsigned long long*>(r.ew)[w] : 0ull;
  }
  __syncthreads();
  auto publish_token = [&](int t, float my_val, int my_idx, float vmax) {
    const float w = routing_weight(my_val, vmax, lane, k, r.sigmoid);
    if (lane < k) {
      reinterpret_cast<float2*>(o.pairs)[(size_t)t * k + lane] = make_float2((float)my_idx, w);
      o.ids[t * k + lane] = my_idx;
      s.ids[t * k + lane] = my_idx;
      s.wts[t * k + lane] = w;
    }
  };
  // a wave's tokens four at a time: their logits are requested together, so that a wave
  // with several tokens waits for memory once
  for (int t0 = wv; t0 < T; t0 += 4 * NW) {
    float v[4][4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int t = t0 + q * NW;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int e = lane + 64 * j;
        v[q][j] = (t < T && e < E) ? r.logits[(size_t)t * E + e] : NEG;
      }
    }
#pragma unroll 1  // one copy of the selection code: the token in turn sits in v[0], the others move up
    for (int q = 0; q < 4; ++q) {
      const int t = t0 + q * NW;
      if (t < T) {
        float my_val, vmax;
        int my_idx;
        bool close_call;
        select_topk(v[0], lane, E, k, my_val, my_idx, vmax, close_call, tol);
        if (close_call) {
          float lo, hi;
          close_call_range(my_val, lane, E, k, tol, lo, hi);
          if (lane == 0) {
            const int n = atomicAdd(&s.cc_n, 1);
            s.cc_tok[n] = t;
            s.cc_lo[n] = lo, s.cc_hi[n] = hi;
          }
        } else {
          publish_token(t, my_val, my_idx, vmax);
        }
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) v[0][j] = v[1][j], v[1][j] = v[2][j], v[2][j] = v[3][j];
    }
  }
#pragma unroll
  for (int i = 0; i < kEwPerThread; ++i) {
    const int w = threadIdx.x + i * NT;
    if (w < kEwWords) s.ew[w] = ew_reg[i];
  }
  __syncthreads();
  // rare: tokens with a close call among their k+1 largest logits are recomputed in the
  // reference's order by the whole workgroup, one after the other; wave 0 selects again
  for (int n = 0; n < s.cc_n; ++n) {
    const int t = s.cc_tok[n];
    logits_reference_order_wg(r.x + (size_t)t * r.H, r.g, r.b, r.logits + (size_t)t * E, E, r.H, s.cc_lo[n], s.cc_hi[n],
                              s.cc);
    if (wv == 0) {
      float v[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int e = lane + 64 * j;
        v[j] = e < E ? s.cc.fixed[e] : NEG;
      }
      float my_val, vmax;
      int my_idx;
      bool close_call;
      select_topk(v, lane, E, k, my_val, my_idx, vmax, close_call, 0.0f);
      publish_token(t, my_val, my_idx, vmax);
    }
    __syncthreads();
  }
  __syncthreads();
  // Dispatch in O(P): thread p owns assignment p.  A chunk's assignments mark themselves in the word of the expert that they
  // name: its bits below a lane's own are the lane's rank there, and a prefix over the chunks gives every assignment its
  // place in the expert's list: assignments stay in ascending order, as the
  // reference's per-expert token loop visits them (expert_mlp_node.h:503-529).
  const int my_p = threadIdx.x;
  const bool live_p = my_p < P;
  const int my_id = live_p ? s.ids[my_p] : 0;
  if (live_p) atomicOr(&s.named[wv][my_id], 1ull << lane);
  __syncthreads();
  for (int e = threadIdx.x; e < E; e += NT) {
    int run = 0;
    for (int c = 0; c < nchunk; ++c) {
      s.before[c][e] = (short)run;
      run += __popcll(s.named[c][e]);
    }
    s.cnt[e] = run;
    o.counts[e] = run;
  }
  __syncthreads();
  // exclusive scan, active experts, list entries: wave 0, four consecutive
  // experts per lane, wave-wide prefix sums
  const int per = r.lists == kListGroups ? r.group_tokens : 64;  // tokens per list entry
  if (wv == 0) {
    int c[4], tot = 0, nact = 0, nent = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int e = lane * 4 + j;
      c[j] = e < E ? s.cnt[e] : 0;
      tot += c[j];
      nact += c[j] > 0;
      nent += group_count(c[j], per);
    }
    // inclusive scans over the lanes, two 16-bit counts to a register (none exceeds MAXP)
    const int sa = wave_scan_inclusive(tot | (nent << 16), lane), s_act = wave_scan_inclusive(nact, lane);
    const int s_tot = sa & 0xffff, s_ent = sa >> 16;
    int run = s_tot - tot, slot = s_act - nact, li = s_ent - nent;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int e = lane * 4 + j;
      if (e < E) {
        s.off[e] = run;
        o.offsets[e] = run;
        s.first[e] = li;
        s.slot[e] = slot;
        if (c[j] > 0) s.act_e[slot++] = e;
        li += group_count(c[j], per);
        run += c[j];
      }
    }
    if (lane == 63) {
      s.na = s_act;
      o.offsets[E] = s_tot;
      *o.nv = r.lists == kListGroups ? s_ent : 0;
      *o.n_mtiles = r.lists == kListGroups ? 0 : s_ent;
    }
  }
  __syncthreads();
  // place of assignment p: the expert's offset + its assignments in earlier chunks + its rank in this one; the first of
  // every list entry's assignments writes the entry
  if (live_p) {
    const unsigned inv_k = (65536u + (unsigned)k - 1u) / (unsigned)k;  // p / k == p * inv_k >> 16 for p <= 1024, k <= 16
    const int rank = s.before[wv][my_id] + __popcll(s.named[wv][my_id] & ((1ull << lane) - 1ull));
    const int pos = s.off[my_id] + rank;
    o.list_tok[pos] = (int)(((unsigned)my_p * inv_k) >> 16);
    o.list_w[pos] = s.wts[my_p];
    o.pos_of_slot[my_p] = pos;
    const int nth = group_count(rank, per);
    if (nth * per == rank) {
      if (r.lists == kListGroups) {
        write_stream_group(o.groups + s.first[my_id] + nth, reinterpret_cast<const ExpertW*>(s.ew) + my_id, my_id,
                           s.cnt[my_id] - rank, pos);
      } else {
        o.mtiles[2 * (s.first[my_id] + nth)] = s.slot[my_id];
        o.mtiles[2 * (s.first[my_id] + nth) + 1] = rank;
      }
    }
  }
  if (r.lists == kListDesc) {
    for (int i = threadIdx.x; i < E; i += NT) {
      const bool on = i < s.na;
      const int e = on ? s.act_e[i] : 0;
      write_work_desc(o.desc + i, on, e, s.cnt[e], s.off[e], reinterpret_cast<const ExpertW*>(s.ew)[e]);
    }
  }
}
}  // namespace csk
