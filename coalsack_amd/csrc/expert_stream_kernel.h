// Expert MLP for the weight-streaming (decode) regime.
//
// Every active expert's matrices are streamed from HBM once per group of up to
// four of its tokens (batches with more per expert take tiles, expert_prefill_kernel.h): 64 lanes x 16 bytes = 1 KiB of contiguous nibbles per
// 16-row tile per K step, the four waves of a workgroup taking interleaved K
// steps (128 elements each).  The MXFP4 entries are the B operand of the block-scaled
// matrix instruction as they are stored, their E8M0 bytes its scale operand; the group's
// activation rows are its A operand as three FP6 terms (mx3.h), so each product is that of
// the reference's fp32 activation (to 2^-14.7 of its block's maximum) and the exactly
// dequantised weight; accumulation is fp32.  The K slices of the four waves meet in LDS in
// a fixed order.
//
// Restates include/coalsack/nn/nn_ops/expert_mlp_node.h:651-732
// (compute_token_mxfp4): gate/up projections + bias, activation (:699-706),
// down projection + bias; the token loop of :503-529 becomes the M dimension.
#pragma once
#include "common.h"
#include "mx3.h"
#include "route_select.h"

namespace csk {

// Bias pointers inside desc[].w must not be null for expert_stream_kernel: the
// host substitutes a zero vector for an absent bias, so that the loads are
// unconditional.
struct ExpertStreamArgs {
  const WorkDesc* desc;
  const StreamGroup* groups;  // [nv]: the groups of up to G tokens
  const int* nv;         // number of such groups
  int nv_known;          // > 0: the number of groups is known at launch (one token: its k experts), *nv is not read
  const int* list_row;   // packed position -> row of X; null: row = packed position
  const float* gather_w; // packed position -> factor applied to its row (weight_before_ffn); null: 1
  const float* X;        // [rows][32 nblk] fp32 activation rows
  const u32x4* X3;       // the same rows already as three FP6 terms, [rows][mx3_row_blocks(nblk)][6] (mx3.h), or null
  const float* zeros;    // at least 16 bytes of zeros (with X3)
  int group_tokens;      // tokens per group: what the groups were formed with
  int nblk;              // K / 32
  int ntile;             // ceil(N / 16)
  int N;                 // output features (F for gate/up, H for down)
  int act_type;
  float* act_out;        // gate/up: [P][N] fp32
  float* y_out;          // down: [P][N] fp32
  RouteIn rin;           // ROUTE1 form only: what the token is routed from ...
  RouteOut rout;         // ... and where workgroup 0 leaves the router's output and the lists
};

// exp and the reciprocal are the hardware's own approximations (v_exp_f32 on x log2 e,
// v_rcp_f32: one ulp each, a relative error near 1e-6 after the argument's rounding at
// |x| <= 12), not libm's expf and an IEEE division: the epilogue of the grouped GEMM
// evaluates 64 of these per lane and was spending more vector instructions on them than
// on anything else.  Both regimes use this one function, so they agree with each other.
__device__ __forceinline__ float fast_sigmoid_mul(float x, float slope) {  // x * sigmoid(slope x)
  const float e = __builtin_amdgcn_exp2f(x * (-slope * 1.4426950408889634f));
  return x * __builtin_amdgcn_rcpf(1.0f + e);
}
__device__ __forceinline__ float moe_activation(float gate_v, float up_v, int act_type) {
  if (act_type == 0) {  // expert_mlp_node.h:699-703
    const float x = fminf(gate_v, 7.0f);
    const float y = fminf(fmaxf(up_v, -7.0f), 7.0f);
    return fast_sigmoid_mul(x, 1.702f) * (y + 1.0f);
  }
  return fast_sigmoid_mul(gate_v, 1.0f) * up_v;  // :705-706
}

// ---------------------------------------------------------------------------
// Persistent, software-pipelined kernel (K <= 8192) on the block-scaled matrix
// instruction v_mfma_scale_f32_16x16x128_f8f6f4: A = the group's activation rows as
// three FP6 terms (mx3.h), B = the MXFP4 weights exactly as they are stored -- lane
// (g = lane / 16, n = lane % 16) holds K block g of the step of weight row n, which is the
// 16-byte entry the repacked plane keeps for it, and passes that block's E8M0 byte as the
// instruction's scale operand.  No conversion instruction touches a weight.
//
// NS = K steps per wave (4 waves x NS x 128 elements cover K), NT = weight tiles per work
// unit (stream_tiles: together they set the loads in flight).
// MODE 0: a work unit is NT/2 gate tiles and the up tiles of the same features, SwiGLU epilogue.
// MODE 1: a work unit is NT consecutive down tiles.
// ROWS3: the rows arrive as FP6 terms and are only copied.  Without the quantiser and its hundred registers the kernel takes
// 98 to 148 instead of 180 to 220, and the one-token form has three workgroups per compute unit, a place for each of 720
// units of a 2880 x 2880 layer (8 layers, one token 239 -> 235 us, 16 tokens 785 -> 782; three per compute unit change
// nothing for more tokens).
// Up to four tokens are contracted per pass (rows 0..3 of the instruction's 16 token rows; the launch says how many,
// a.group_tokens).
//
// The work is (token group of an expert) x (tile pair): every group costs the
// same, so teams of gridDim.x / groups workgroups take one group each and
// interleave its units, and the load is balanced whatever the routing was.
// Memory-level parallelism bounds this kernel, so it never lets the memory
// queue drain: the weight registers are refilled step by step as the matrix cores
// consume them: the loads of unit t+1 -- issued unconditionally from clamped addresses so
// that no full wait separates them -- are in flight while unit t is contracted, and every wait
// of the unit loop leaves all but the step's own loads in flight.  That takes a wave number
// which the compiler knows to be uniform (or each load sits in a loop over its scalar offset,
// and the wait-count pass drains the queue at the unit's head), scale bytes requested in front of the
// weights, and matrix instructions pinned between the refills.  Measured against the form with
// none of these: one token through 8 layers of 2880 x 2880 251 -> 238 us, 64 experts of 2048 x 768,
// 50 tokens, 8 layers, 628 -> 602 us, a two-token host frame 60 -> 57 us.  A
// group's activation rows arrive as fp32 and are quantised to the three-term form by the
// workgroup itself, into LDS, while its first weight loads are under way.  The four waves
// split K; their partial sums meet in double-buffered LDS (one barrier per unit) in the
// fixed order w0 + w1 + w2 + w3, and wave t mod 4 finishes unit t.
typedef int i32x8 __attribute__((ext_vector_type(8)));

// A close call of the one token: eight logits side by side, their products staged in pieces of half the length, so that the
// staging area leaves room for three workgroups per compute unit.  (Four of them in whole pieces take as much LDS, but top-4
// has at least five to recompute, one chain of dependent additions after the other in every workgroup.  8 layers of 2880 x
// 2880, top-4, with a close call in each: four at a time 455 us, in pieces of 512 357, of 384 353; without any 237, and 239.5 with
// pieces of 512, whose code is longer.)
using RouteOneLds = CloseCallLdsT<256, kCcBatch, kCcChunk / 2>;
constexpr int kRouteOneWgPerCu = 3;
static_assert(kRouteOneWgPerCu * (sizeof(RouteOneLds) + kMaxExperts * sizeof(ExpertW) + 1280) <= 160 * 1024,
              "the staging area beside the pointer table, allocated in units of 1280 bytes");
// Descriptor of a whole weight plane as a raw buffer (the pointer is the same in every lane).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t stream_plane_rsrc(const void* p) {
  const uint64_t v = reinterpret_cast<uint64_t>(p);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)v);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(v >> 32));
  return __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<char*>(((uint64_t)hi << 32) | lo), 0, 0x7fffffff, 0x00020000);
}

//
// ROUTE = 1 (gate/up of a one-token batch): there is no routing kernel in front.  Every
// workgroup selects the token's k experts itself from the logits -- select_topk in each of
// its four waves, so that nothing passes from wave to wave; a close call recomputed by the
// whole workgroup, exactly as route_tiny_kernel does; all workgroups compute the same thing
// from the same inputs -- and takes the expert whose rank among the selected ones is its
// team's number: that rank is the expert's packed position, as the dispatch would have
// numbered it.  The experts' pointer table is staged in LDS while the logits are on their
// way.  Workgroup 0 also writes what the routing kernel would have written (pairs, ids,
// positions, lists, counts, token groups) for the down kernel, the combine and
// csk_layer_last_dispatch.  A 5.4 us launch with its dependent reads is replaced by 3 us in
// front of this kernel's first weight loads (120b shape: 32.6 -> 30.0 us per layer).
//
// ROUTE = kRouteFewTokens (gate/up of up to eight tokens with at most 64 assignments): the same for a few tokens.  Wave w
// selects for tokens w and w + 4, the selections meet in LDS, and from there each wave places all of them, an assignment
// per lane, as route_tiny_kernel does; the workgroup's token group, its place and its tokens then come out of ballots, and
// how many groups there are, which the teams go by, is known only here (8 layers of 2880 x 2880, 2 tokens 317 -> 290 us, of which a
// launch and its dependent reads are 27; a two-token host frame 54.6 -> 51.5).
//
// Shape of a work unit.  Twelve or more 1 KiB weight loads in flight per wave keep the memory
// system busy; a K of 2880 gives that from two tiles of six steps, a shorter one walks fewer
// steps (a K of 768 used to walk six, four of them past the end of K) and takes four tiles,
// a longer one more steps.  Measured: 64 experts of 2048 x 768, 50 tokens x top-8, down kernel
// 40.5 -> 22.0 us, gate/up 34.0 -> 29.1; 16 experts of 4096 x 6144, 6 tokens, which the grouped GEMM
// used to take (62 + 65 us): 52 + 29.  Tiles per unit: with two everywhere the first case's down kernel
// takes 23.8 us, with six at two steps 23 us and more; at twelve and sixteen steps two down tiles
// beat one by 2 to 3 % of the layer, and at six steps one tile loses 6 %.
constexpr int kStreamMaxBlocks = 256;  // K / 32
constexpr int stream_steps(int nblk) {  // K steps per wave, of the forms that are instantiated
  const int ns = (nblk + 15) / 16;
  return ns <= 2 ? 2 : ns <= 6 ? ns : ns <= 8 ? 8 : ns <= 12 ? 12 : 16;
}
constexpr int stream_tiles(int ns) {
  return ns <= 3 ? 4 : 2;
}
constexpr int stream_depth(int ns) { return ns <= 8 ? ns : ns / 2; }  // divides ns: a step's registers are known at compile time
constexpr size_t stream_lds_bytes(int ns, int group_tokens) {
  // activation rows as three FP6 terms (96 B per block, 16 ns blocks per row: zeros past K) + the reduction buffers
  return (size_t)group_tokens * ns * 16 * 96 + (size_t)2 * 4 * (4 * stream_tiles(ns)) * 16 * sizeof(float);
}

template <int MODE, int NS, int ROUTE = 0, bool ROWS3 = false>
__global__ __launch_bounds__(256, ROUTE == 1 && ROWS3 ? kRouteOneWgPerCu : 2) void expert_stream_kernel(ExpertStreamArgs a) {
  static_assert(ROUTE == 0 || MODE == 0, "the gate/up kernel is the one that routes");
  static_assert(ROUTE <= 1 || (ROUTE == kRouteFewTokens && ROWS3), "several tokens: rows that are only copied");
  constexpr bool ROUTE1 = ROUTE == 1;
  constexpr int NT = stream_tiles(NS);  // weight tiles per unit
  constexpr int TU = MODE == 0 ? NT / 2 : NT; // tiles of one plane per unit
  constexpr int ND = stream_depth(NS);        // K steps whose weights are held or in flight
  constexpr int NV = 4 * NT;                  // accumulator floats per lane per unit
  constexpr int G = kStreamG;                 // tokens per pass, at most
  extern __shared__ __align__(16) unsigned char smem[];
  const int nblk = a.nblk;
  // blocks per activation row in LDS: all the blocks the steps touch, those past K zero, so
  // that nothing in the main loop is clamped or masked (weight blocks past K are then the
  // next tile's, or the slack behind the plane, times exact zeros)
  constexpr int lrb = NS * 16;
  u32x4* As = reinterpret_cast<u32x4*>(smem);  // [group_tokens][lrb][3 terms][2] x 16 B
  float* red = reinterpret_cast<float*>(smem + (size_t)a.group_tokens * lrb * (kMx3ChunksPerBlock * 16));  // [2][4][NV][16]: live lanes only

  const int npair = (a.ntile + TU - 1) / TU;  // units per token group
  // Teams of W workgroups share one token group and interleave its units
  // (workgroup j takes units j, j + W, ...), so that at any moment a team reads one
  // contiguous window of the expert's planes.
  int nvv = 0, W = 1, teams = 1, team = 0, tj = 0;
  auto take_place = [&](int groups) {  // false: no work for this workgroup
    nvv = groups;
    W = max(1, (int)gridDim.x / max(nvv, 1));
    teams = gridDim.x / W;
    team = blockIdx.x / W, tj = blockIdx.x % W;
    return team < teams && tj < npair;
  };
  if constexpr (ROUTE <= 1) {
    if (!take_place(a.nv_known > 0 ? a.nv_known : *a.nv)) return;  // (known: one dependent read fewer in front of the first weights)
  }
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // wave-uniform, and known to be: it is part of the weight loads' scalar offsets
  const int n = lane & 15, g = lane >> 4;

  // ROUTE1: slot s of the token in lane s of every wave (all four waves select, from the same
  // logits, so that nothing has to be handed from wave to wave)
  int r_idx = 0;
  float r_wt = 0.0f;
  constexpr int kEwWords = kMaxExperts * (int)(sizeof(ExpertW) / 8), kEwPerThread = (kEwWords + 255) / 256;
  __shared__ unsigned long long s_ew[ROUTE ? kEwWords : 1];  // the experts' weight pointers, staged beside the logits
  if constexpr (ROUTE1) {
    const RouteIn& r = a.rin;
    const int E = r.E, k = r.k;
    // the recomputation's staging area lies where the activation rows go afterwards
    RouteOneLds& cc = *reinterpret_cast<RouteOneLds*>(smem);
    const float NEG = -__builtin_inff();
    float v[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int e = lane + 64 * j;
      v[j] = e < E ? r.logits[e] : NEG;
    }
    unsigned long long ew_reg[kEwPerThread];
#pragma unroll
    for (int i = 0; i < kEwPerThread; ++i) {
      const int w = threadIdx.x + i * 256;
      ew_reg[i] = w < E * (int)(sizeof(ExpertW) / 8) ? reinterpret_cast<const unsigned long long*>(r.ew)[w] : 0ull;
    }
    float my_val, vmax;  // lane s keeps slot s
    bool close_call;
    const float tol = close_call_tolerance(r.H);
    select_topk(v, lane, E, k, my_val, r_idx, vmax, close_call, tol);
#pragma unroll
    for (int i = 0; i < kEwPerThread; ++i) {
      const int w = threadIdx.x + i * 256;
      if (w < kEwWords) s_ew[w] = ew_reg[i];
    }
    if (close_call) {  // the same in every wave, and in every workgroup
      float lo, hi;
      close_call_range(my_val, lane, E, k, tol, lo, hi);
      logits_reference_order_wg(r.x, r.g, r.b, r.logits, E, r.H, lo, hi, cc);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int e = lane + 64 * j;
        v[j] = e < E ? cc.fixed[e] : NEG;
      }
      select_topk(v, lane, E, k, my_val, r_idx, vmax, close_call, 0.0f);
    }
    r_wt = routing_weight(my_val, vmax, lane, k, r.sigmoid);
    __syncthreads();  // the pointer table is in LDS; every thread is done with cc before the activation rows overwrite it
    if (blockIdx.x == 0) {
      // what the routing kernel would have written (where to: read from the arguments here -- left to the compiler the addresses
      // are read in every workgroup and held in scalar registers over all that comes before)
      auto args = (const __attribute__((address_space(4))) ExpertStreamArgs*)__builtin_amdgcn_kernarg_segment_ptr();
      asm volatile("" : "+s"(args));
      const auto& o = args->rout;
      __shared__ int w_ids[kMaxTopK];
      if (wv == 0 && lane < k) w_ids[lane] = r_idx;
      __syncthreads();
      for (int e = threadIdx.x; e < E; e += 256) {
        int c = 0;
        for (int q = 0; q < k; ++q) c += w_ids[q] == e;
        o.counts[e] = c;
      }
      if (wv == 0 && lane < k) {
        int pos = 0;
        for (int q = 0; q < k; ++q) pos += w_ids[q] < r_idx;  // the k experts are distinct
        reinterpret_cast<float2*>(o.pairs)[lane] = make_float2((float)r_idx, r_wt);
        o.ids[lane] = r_idx;
        o.list_tok[pos] = 0;
        o.list_w[pos] = r_wt;
        o.pos_of_slot[lane] = pos;
        write_stream_group(o.groups + pos, reinterpret_cast<const ExpertW*>(s_ew) + r_idx, r_idx, 1, pos);
      }
      if (threadIdx.x == 0) *o.nv = k;
    }
  }

  // ROUTE > 1: assignment p = token * k + slot in lane p of every wave
  int r_lower = 0, r_same = 0, r_before = 0;  // assignments of lower experts, of its own, and of its own from earlier tokens
  int r_group = 0;                            // token groups in front of the one that it begins ...
  bool r_first = false;                       // ... if it begins one
  if constexpr (ROUTE > 1) {
    const RouteIn& r = a.rin;
    const int E = r.E, k = r.k, T = r.T, P = T * k;
    RouteOneLds& cc = *reinterpret_cast<RouteOneLds*>(smem);
    __shared__ int s_ids[kRouteTinyMaxP], s_cc[kRouteFewTokens];
    __shared__ float s_wt[kRouteTinyMaxP], s_lo[kRouteFewTokens], s_hi[kRouteFewTokens];
    const float NEG = -__builtin_inff();
    constexpr int kTurns = kRouteFewTokens / 4;  // wave w selects for tokens w, w + 4, ...
    float v[kTurns][4];
#pragma unroll
    for (int q = 0; q < kTurns; ++q) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int t = wv + 4 * q, e = lane + 64 * j;
        v[q][j] = t < T && e < E ? r.logits[(size_t)t * E + e] : NEG;
      }
    }
    unsigned long long ew_reg[kEwPerThread];
#pragma unroll
    for (int i = 0; i < kEwPerThread; ++i) {
      const int w = threadIdx.x + i * 256;
      ew_reg[i] = w < E * (int)(sizeof(ExpertW) / 8) ? reinterpret_cast<const unsigned long long*>(r.ew)[w] : 0ull;
    }
    const float tol = close_call_tolerance(r.H);
    auto publish = [&](int t, float my_val, int my_idx, float vmax) {
      const float w = routing_weight(my_val, vmax, lane, k, r.sigmoid);
      if (lane < k) s_ids[t * k + lane] = my_idx, s_wt[t * k + lane] = w;
    };
    bool close_any = false;
#pragma unroll 1  // one copy of the selection code: the token in turn sits in v[0], the others move up
    for (int t = wv; t < T; t += 4) {
      float my_val, vmax;
      int my_idx;
      bool close_call;
      select_topk(v[0], lane, E, k, my_val, my_idx, vmax, close_call, tol);
      if (lane == 0) s_cc[t] = close_call;
      if (close_call) {
        float lo, hi;
        close_call_range(my_val, lane, E, k, tol, lo, hi);
        if (lane == 0) s_lo[t] = lo, s_hi[t] = hi;
        close_any = true;
      } else {
        publish(t, my_val, my_idx, vmax);
      }
#pragma unroll
      for (int q = 0; q + 1 < kTurns; ++q)
#pragma unroll
        for (int j = 0; j < 4; ++j) v[q][j] = v[q + 1][j];
    }
#pragma unroll
    for (int i = 0; i < kEwPerThread; ++i) {
      const int w = threadIdx.x + i * 256;
      if (w < kEwWords) s_ew[w] = ew_reg[i];
    }
    if (__syncthreads_or(close_any)) {
      for (int t = 0; t < T; ++t) {
        if (!s_cc[t]) continue;
        logits_reference_order_wg(r.x + (size_t)t * r.H, r.g, r.b, r.logits + (size_t)t * E, E, r.H, s_lo[t], s_hi[t], cc);
        if (wv == 0) {
          float vt[4], my_val, vmax;
          int my_idx;
          bool close_call;
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const int e = lane + 64 * j;
            vt[j] = e < E ? cc.fixed[e] : NEG;
          }
          select_topk(vt, lane, E, k, my_val, my_idx, vmax, close_call, 0.0f);
          publish(t, my_val, my_idx, vmax);
        }
        __syncthreads();
      }
    }
    const bool lp = lane < P;
    r_idx = lp ? s_ids[lane] : 0x7fffffff;
    for (int q = 0; q < P; ++q) {  // q is the same in every lane
      const int idq = __builtin_amdgcn_readlane(r_idx, q);
      r_lower += idq < r_idx;
      r_same += idq == r_idx;
      r_before += idq == r_idx && q < lane;
    }
    r_first = lp && r_before % G == 0;
    const unsigned long long firsts = __ballot(r_first);
    for (unsigned long long m = firsts; m != 0ull; m &= m - 1ull) {
      const int q = (int)__builtin_ctzll(m), idq = __builtin_amdgcn_readlane(r_idx, q);
      r_group += idq < r_idx || (idq == r_idx && q < lane);
    }
    if (blockIdx.x == 0) {
      // what the routing kernel would have written (see the one-token form for where to)
      auto args = (const __attribute__((address_space(4))) ExpertStreamArgs*)__builtin_amdgcn_kernarg_segment_ptr();
      asm volatile("" : "+s"(args));
      const auto& o = args->rout;
      for (int e = threadIdx.x; e < E; e += 256) {
        int c = 0;
        for (int q = 0; q < P; ++q) c += s_ids[q] == e;
        o.counts[e] = c;
      }
      if (wv == 0 && lp) {
        const int pos = r_lower + r_before;
        const unsigned inv_k = (65536u + (unsigned)k - 1u) / (unsigned)k;  // p / k == p * inv_k >> 16 for p < 64, k <= 16
        reinterpret_cast<float2*>(o.pairs)[lane] = make_float2((float)r_idx, s_wt[lane]);
        o.ids[lane] = r_idx;
        o.list_tok[pos] = (int)(((unsigned)lane * inv_k) >> 16);
        o.list_w[pos] = s_wt[lane];
        o.pos_of_slot[lane] = pos;
        if (r_first) write_stream_group(o.groups + r_group, reinterpret_cast<const ExpertW*>(s_ew) + r_idx, r_idx, r_same - r_before, pos);
        if (lane == 0) *o.nv = __popcll(firsts);
      }
    }
    if (!take_place(__popcll(firsts))) return;
  }

  // a lane's scale bytes of one tile: 2, 4, 8 or 16, one per step of the wave rounded up (scale_slots)
  constexpr int kScWords = NS <= 4 ? 1 : NS <= 8 ? 2 : 4;
  typedef uint32_t ScaleWords __attribute__((ext_vector_type(kScWords)));
  using ScaleCell = std::conditional_t<NS == 2, uint16_t, ScaleWords>;
  struct WSet {
    u32x4 q[ND][NT];
    ScaleWords sc[NT];  // this wave's scale bytes of the tiles, one byte per K step
    float b[NT];
  };

  int par = 0;
  for (int v = team; v < nvv; v += teams) {
    const int p_begin = tj, p_end = npair;
    const StreamGroup* gr = a.groups + v;
    int r_e = 0;
    float r_gw = 1.0f;
    if constexpr (ROUTE1) {  // the selected expert with v selected experts below it: packed position v
      const int k = a.rin.k;
      int lower = 0;
      for (int q = 0; q < k; ++q) lower += __builtin_amdgcn_readlane(r_idx, q) < r_idx;
      const unsigned long long mine = __ballot(lane < k && lower == v);
      const int sl = (int)__builtin_ctzll(mine | (1ull << 63));
      r_e = __builtin_amdgcn_readlane(r_idx, sl);
      r_gw = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(r_wt), sl));
    }
    int r_base = 0, r_count = 0;
    int r_tok[G] = {};
    if constexpr (ROUTE > 1) {  // the group with v groups before it, and its tokens: the assignments that name its expert
      const int sl = (int)__builtin_ctzll(__ballot(r_first && r_group == v) | (1ull << 63));
      const int skip = __builtin_amdgcn_readlane(r_before, sl);
      r_e = __builtin_amdgcn_readlane(r_idx, sl);
      r_base = __builtin_amdgcn_readlane(r_lower, sl) + skip;
      r_count = min(G, __builtin_amdgcn_readlane(r_same, sl) - skip);
      const unsigned inv_k = (65536u + (unsigned)a.rin.k - 1u) / (unsigned)a.rin.k;
      unsigned long long named = __ballot(r_idx == r_e && r_before >= skip);
#pragma unroll
      for (int i = 0; i < G; ++i) {
        r_tok[i] = named != 0ull ? (int)(((unsigned)__builtin_ctzll(named) * inv_k) >> 16) : r_tok[i > 0 ? i - 1 : 0];
        named &= named - 1ull;
      }
    }
    const ExpertW* gw_ptr = ROUTE ? reinterpret_cast<const ExpertW*>(s_ew) + r_e : &gr->w;
    const int gcount = ROUTE1 ? 1 : ROUTE ? r_count : min(a.group_tokens, gr->left);
    const int base = ROUTE1 ? v : ROUTE ? r_base : gr->base;
    // One buffer descriptor per weight plane: the unit's tile and the K step go into the
    // scalar offset of a load, the lane's place within the step (block g, row n) into its
    // vector offset, which never changes.
    const auto q_rsrc0 = stream_plane_rsrc(MODE == 0 ? gw_ptr->q_gate : gw_ptr->q_down);
    const auto q_rsrc1 = stream_plane_rsrc(MODE == 0 ? gw_ptr->q_up : gw_ptr->q_down);
    const uint32_t qoff = (uint32_t)((g * 16 + n) * 16);
    const CSK_GLOBAL ScaleCell* s0 = as_global(reinterpret_cast<const ScaleCell*>(MODE == 0 ? gw_ptr->s_gate : gw_ptr->s_down)) + wv * 64 + lane;
    const CSK_GLOBAL ScaleCell* s1 = as_global(reinterpret_cast<const ScaleCell*>(MODE == 0 ? gw_ptr->s_up : gw_ptr->s_down)) + wv * 64 + lane;
    const CSK_GLOBAL float* bp0 = as_global(MODE == 0 ? gw_ptr->b_gate : gw_ptr->b_down);
    const CSK_GLOBAL float* bp1 = as_global(MODE == 0 ? gw_ptr->b_up : gw_ptr->b_down);

    // Tile m of a unit: gate tiles TU unit .. then the up tiles of the same features, or down
    // tiles NT unit ..; past the last tile the last one again (its results are dropped).
    auto tile_of = [&](int unit, int m) { return min(unit * TU + m % TU, a.ntile - 1); };
    // `idle`: a refill whose data nobody will use (past the workgroup's last unit).  It is
    // still issued, so that the count of loads in flight is the same on every path, but
    // every step aims at the same 1 KiB of the unit, which the caches hold: the tail of a
    // workgroup must not cost HBM traffic.
    auto load_step = [&](WSet& ws, int unit, int s, bool idle) {
      // four blocks of 16 rows x 16 B per step; a step that lies wholly past K (its activations
      // are zeros) re-reads the cached start of the tile instead of fetching the next tile's blocks
      const uint32_t step = (idle || 4 * (wv + 4 * s) >= nblk) ? 0u : (uint32_t)(wv + 4 * s) * 1024u;
#pragma unroll
      for (int m = 0; m < NT; ++m)
        ws.q[s % ND][m] = __builtin_amdgcn_raw_buffer_load_b128(m < TU ? q_rsrc0 : q_rsrc1, qoff,
                                                           (uint32_t)tile_of(unit, m) * (uint32_t)nblk * 256u + step, 0);
    };
    // per-unit scalars: the wave's scale bytes (scale plane: [tile][wave][lane][slots]) and biases
    auto load_unit_scalars = [&](WSet& ws, int unit) {
#pragma unroll
      for (int m = 0; m < NT; ++m) {
        const int t = tile_of(unit, m);
        if constexpr (NS == 2) ws.sc[m][0] = (m < TU ? s0 : s1)[(size_t)t * 256];
        else ws.sc[m] = (m < TU ? s0 : s1)[(size_t)t * 256];
        ws.b[m] = (m < TU ? bp0 : bp1)[min(t * 16 + n, a.N - 1)];  // bias pointers are never null (absent bias = zero vector)
      }
    };
    const bool live = g == 0;  // token t is accumulator row t of the first sixteen lanes

    // A thread's first block of activations is requested first (loads return in order: asked
    // for after the weights it would arrive behind them), then the first unit's weights ...
    const int nfill = gcount * lrb;
    // Rows that arrive as FP6 terms already (written once per token by the routing prologue)
    // are only copied into LDS, behind the first unit's weights (below).
    constexpr bool copy_rows = ROWS3;
    int copy_row[G];  // the rows' numbers, read before the weights are requested
    if (copy_rows) {
#pragma unroll
      for (int rr = 0; rr < G; ++rr) {
        const int p = base + min(rr, gcount - 1);
        copy_row[rr] = ROUTE1 ? 0 : ROUTE ? r_tok[rr] : a.list_row ? a.list_row[p] : p;
      }
    }
    float4 pre[8];
    if constexpr (!ROWS3) {
      const int rr = threadIdx.x / lrb, kb = threadIdx.x - rr * lrb;
      if ((int)threadIdx.x < nfill && kb < nblk) {
        const int row = ROUTE1 ? 0 : a.list_row ? a.list_row[base + rr] : base + rr;
        const float4* src = reinterpret_cast<const float4*>(a.X + ((size_t)row * nblk + kb) * 32);
#pragma unroll
        for (int i = 0; i < 8; ++i) pre[i] = src[i];
      }
    }
    WSet ws;
    load_unit_scalars(ws, p_begin);
#pragma unroll
    for (int s = 0; s < ND; ++s) load_step(ws, p_begin, s, false);

    // ... and while those are under way the group's activation rows are
    // quantised into LDS, one thread per 32-value block (every wave is past its last read
    // of the previous group: it has crossed that unit's barrier).  Rows may be gathered
    // through list_row and scaled by the routing weight (weight_before_ffn).
    if constexpr (ROWS3) {
      // The LDS image of a row is its blocks in order, [lrb][6 chunks of 16 bytes]; the row in
      // memory has mx3_row_blocks(nblk) of them, the rest are zeros (any scale byte will do
      // for a block of zero codes: they come from the library's page of zeros).  Copied by
      // global_load_lds -- nothing of it lives in a register; instruction i of wave wv fills
      // the 64 chunks from (4 i + wv) * 64 on -- and waited for explicitly: the compiler does
      // not count these loads, so none of them may be in flight past the wait below.
      const int rowblk = mx3_row_blocks(nblk);
      constexpr int kRowChunks = lrb * kMx3ChunksPerBlock;
      const int total = gcount * kRowChunks;
      const uint32_t lds_as = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)smem;
#pragma unroll 1
      for (int i = 0; i * 256 < total; ++i) {
        const int ch0 = (4 * i + wv) * 64;
        const int ch = ch0 + lane;
        if (ch < total) {
          const int rr = ch / kRowChunks, q = ch - rr * kRowChunks;
          int row = copy_row[0];
#pragma unroll
          for (int x = 1; x < G; ++x) row = rr == x ? copy_row[x] : row;
          const u32x4* src = q < rowblk * kMx3ChunksPerBlock ? a.X3 + (size_t)row * rowblk * kMx3ChunksPerBlock + q
                                                            : reinterpret_cast<const u32x4*>(a.zeros);
          asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off"
                       :
                       : "v"(src), "s"(__builtin_amdgcn_readfirstlane((int)(lds_as + (uint32_t)ch0 * 16u)))
                       : "memory");
        }
      }
      __builtin_amdgcn_s_waitcnt((7 << 4) | (15 << 8));  // vmcnt(0): the copies (and the first weights) have landed
    }
    if constexpr (!ROWS3) {
#pragma unroll 1
    for (int idx = threadIdx.x; idx < nfill; idx += 256) {
      const int rr = idx / lrb, kb = idx - rr * lrb;
      u32x4 out[kMx3ChunksPerBlock];
      if (kb >= nblk) {
#pragma unroll
        for (int t = 0; t < kMx3Terms; ++t) {
          out[2 * t] = u32x4{0u, 0u, 0u, 0u};
          out[2 * t + 1] = u32x4{0u, 0u, 127u, 0u};
        }
      } else {
        float r[32];
        if (idx != (int)threadIdx.x) {  // later blocks of this thread: fetched here
          const int row = ROUTE1 ? 0 : a.list_row ? a.list_row[base + rr] : base + rr;
          const float4* src = reinterpret_cast<const float4*>(a.X + ((size_t)row * nblk + kb) * 32);
#pragma unroll
          for (int i = 0; i < 8; ++i) pre[i] = src[i];
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) r[4 * i] = pre[i].x, r[4 * i + 1] = pre[i].y, r[4 * i + 2] = pre[i].z, r[4 * i + 3] = pre[i].w;
        if (a.gather_w) {
          const float gw = ROUTE1 ? r_gw : a.gather_w[base + rr];  // (the list of weights is being written by workgroup 0)
#pragma unroll
          for (int i = 0; i < 32; ++i) r[i] = r[i] * gw;
        }
        mx3_quantize_block(r, out);
      }
      u32x4* dst = As + (size_t)idx * kMx3ChunksPerBlock;
#pragma unroll
      for (int c = 0; c < kMx3ChunksPerBlock; ++c) dst[c] = out[c];
    }
    }
    // lanes past the group's tokens re-read its last row; their outputs are unused
    const int frag0 = (min(n, gcount - 1) * lrb + 4 * wv + g) * kMx3ChunksPerBlock;

    // Contracts unit `unit` out of ws and, step by step, refills ws with unit `next`.
    auto compute_unit = [&](WSet& ws, int unit, int next) {
      const bool idle = next == unit;
      float bias[NT];
      uint32_t scb[NT][kScWords];
#pragma unroll
      for (int m = 0; m < NT; ++m) {
        bias[m] = ws.b[m];
        asm volatile("" : "+v"(bias[m]));  // (copied before they are overwritten)
#pragma unroll
        for (int w = 0; w < kScWords; ++w) {
          scb[m][w] = ws.sc[m][w];
          asm volatile("" : "+v"(scb[m][w]));
        }
      }
      // in front of the weights: a unit's first matrix instruction needs its scale bytes, and
      // loads retire in order
      load_unit_scalars(ws, next);
      floatx4 acc[NT];  // one 16 x 16 tile each
#pragma unroll
      for (int m = 0; m < NT; ++m) acc[m] = floatx4{0.f, 0.f, 0.f, 0.f};
      u32x4 flo[2], fhi[2];  // activation fragments run one term ahead of the matrix cores
      // The fragments are the same for every unit of the group; unseen by the compiler, which
      // would otherwise read all of them once in front of the unit loop and spill.
      int frag = frag0;
      asm volatile("" : "+v"(frag));
      auto read_frag = [&](int i) {  // fragment i = (step, term)
        const int s = i / kMx3Terms, t = i - s * kMx3Terms;
        const u32x4* f = As + frag + (16 * s * kMx3Terms + t) * 2;  // a constant offset from the lane's base
        flo[i & 1] = f[0];
        fhi[i & 1] = f[1];
      };
      read_frag(0);
#pragma unroll
      for (int s = 0; s < NS; ++s) {
#pragma unroll
        for (int t = 0; t < kMx3Terms; ++t) {
          const int i = s * kMx3Terms + t;
          if (i + 1 < NS * kMx3Terms) read_frag(i + 1);
          // FP6 reads the first six registers; register 6 holds the term's scale byte
          const i32x8 aw = (i32x8)__builtin_shufflevector(flo[i & 1], fhi[i & 1], 0, 1, 2, 3, 4, 5, 6, 7);
#pragma unroll
          for (int m = 0; m < NT; ++m) {
            const int byte = (int)((scb[m][s >> 2] >> (8 * (s & 3))) & 0xFFu);
            const i32x8 bw = (i32x8)__builtin_shufflevector(ws.q[s % ND][m], ws.q[s % ND][m], 0, 1, 2, 3, -1, -1, -1, -1);
            acc[m] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(aw, bw, acc[m], 2, 4, 0, aw[6], 0, byte);
          }
#pragma unroll
          for (int m = 0; m < NT; ++m) asm volatile("" : "+v"(acc[m]));  // the matrix instructions stay on this side of the barrier
          // fragments are read one ahead, not all at once: the scheduler may not hoist the LDS reads over this point
          __builtin_amdgcn_sched_barrier(0);
        }
        // this step's registers are free: start the loads of the step ND further on, in this unit or the next
        if (s + ND < NS) load_step(ws, unit, s + ND, false);
        else load_step(ws, next, s + ND - NS, idle);
      }
      float* rbuf = red + (size_t)par * 4 * NV * 16;
      par ^= 1;
      if (live) {
#pragma unroll
        for (int m = 0; m < NT; ++m)
#pragma unroll
          for (int i = 0; i < 4; ++i) rbuf[(wv * NV + m * 4 + i) * 16 + n] = acc[m][i];
      }
      __syncthreads();
      if (wv == (unit & 3) && live) {
        float v2[NT][4];
#pragma unroll
        for (int m = 0; m < NT; ++m)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int o = m * 4 + i;
            v2[m][i] = ((rbuf[(0 * NV + o) * 16 + n] + rbuf[(1 * NV + o) * 16 + n]) + rbuf[(2 * NV + o) * 16 + n]) +
                       rbuf[(3 * NV + o) * 16 + n];
          }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          if (i < gcount) {
            const size_t p = (size_t)(base + i);  // token i of the group
#pragma unroll
            for (int m = 0; m < TU; ++m) {
              const int r = (unit * TU + m) * 16 + n;  // output feature
              if (r >= a.N) continue;
              if (MODE == 0)
                a.act_out[p * (size_t)a.N + r] = moe_activation(v2[m][i] + bias[m], v2[TU + m < NT ? TU + m : m][i] + bias[TU + m < NT ? TU + m : m], a.act_type);
              else
                a.y_out[p * (size_t)a.N + r] = v2[m][i] + bias[m];
            }
          }
        }
      }
    };

    // One register set, refilled step by step as it is consumed: the loads of unit
    // t+1 are issued during unit t and stay one unit ahead of their use.  Refills
    // are unconditional (past the last unit they re-read one cached KiB of it), so
    // that the number of loads in flight is the same on every path and the waits in
    // front of the matrix cores stay partial.
    const int t_last = p_begin + ((p_end - 1 - p_begin) / W) * W;  // last unit of this workgroup
    __syncthreads();  // the quantised rows are in LDS
    for (int t = p_begin; t < p_end; t += W) compute_unit(ws, t, min(t + W, t_last));
  }
}

// ---------------------------------------------------------------------------
// Down projection and merge of a few tokens in one launch: a workgroup owns NT tiles of 16 output features for all token groups
// of the batch, so that the weighted sum over a token's experts (combine_kernel) needs nothing from another workgroup.
// Its waves are teams of four; a team takes every second or fourth group, its waves split K as those of expert_stream_kernel
// do, and the same partial sums are added in the same order, then weighted and added slot by slot as combine_kernel does: the
// same bits.  The rows of all assignments are quantised into LDS once, beside the first groups' weights on their way:
// those of four groups are requested at the start, by four teams, or by two with two register sets where a row's steps
// take more registers than sixteen waves can have.  A workgroup streams the tiles of all active experts, with one
// workgroup on two compute units of three, so this is for batches whose weights are on their way in one or two
// rounds of latency, of which the launch that the merge needs costs another (8 layers, us, two launches / one: 32
// experts of 2880 x 2880, one token, top-4 230.4 / 218.9, top-2 177 / 163; 64 of 2048 x 768, top-1 141 / 119, top-4 156 / 143; two tokens,
// top-4, eight assignments of 2880 x 2880 290 / 308).
struct ExpertMergeArgs {
  const float* act;  // [P][32 nblk] fp32, by packed position
  const StreamGroup* groups;
  const int* nv;
  int nv_known;      // > 0: the number of groups
  int T, k, nblk, N, ntile;
  const float* pairs;      // [T, k, 2]
  const int* pos_of_slot;  // [T * k]
  const float* residual;   // null: none
  float* out;              // [T, N]
  float2* pairs_out;       // takes a copy of the router output, if given
  int pre_weighted;
};
constexpr int merge_teams(int ns, int nt) { return ns <= 3 && nt == 1 ? 4 : 2; }
constexpr size_t merge_lds_bytes(int ns, int nt, int P) {
  return (size_t)P * ns * 16 * 96 + (size_t)2 * merge_teams(ns, nt) * 4 * 4 * nt * 16 * 4 + (size_t)P * nt * 16 * 4 + (size_t)P * 8;
}

template <int NS, int NT>
__global__ __launch_bounds__(256 * merge_teams(NS, NT)) void expert_stream_kernel_merge(ExpertMergeArgs a) {
  extern __shared__ __align__(16) unsigned char smem[];
  constexpr int kMergeTeams = merge_teams(NS, NT), kMergeThreads = 256 * kMergeTeams, kSets = 4 / kMergeTeams;
  constexpr int ND = stream_depth(NS), lrb = NS * 16, NV = 4 * NT;
  const int P = a.T * a.k, nblk = a.nblk;
  u32x4* const As = reinterpret_cast<u32x4*>(smem);                                               // [P][lrb][3 terms][2]
  float* const red = reinterpret_cast<float*>(smem + (size_t)P * lrb * kMx3ChunksPerBlock * 16);  // [2][teams][4][NV][16]
  float* const ys = red + 2 * kMergeTeams * 4 * NV * 16;                                          // [P][NT * 16]
  int* const s_pos = reinterpret_cast<int*>(ys + P * NT * 16);
  float* const s_wt = reinterpret_cast<float*>(s_pos + P);
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), team = wid >> 2, wv = wid & 3;
  const int n = lane & 15, g = lane >> 4;
  const int nvv = a.nv_known > 0 ? a.nv_known : *a.nv;
  const int tile0 = blockIdx.x * NT;

  // the first block of activations is requested first (loads return in order), then weights
  const int nfill = P * lrb;
  float4 pre[8];
  auto fetch_block = [&](int idx) {
    const int rr = idx / lrb, kb = idx - rr * lrb;
    if (idx < nfill && kb < nblk) {
      const float4* src = reinterpret_cast<const float4*>(a.act + ((size_t)rr * nblk + kb) * 32);
#pragma unroll
      for (int i = 0; i < 8; ++i) pre[i] = src[i];
    }
  };
  fetch_block(threadIdx.x);
  if ((int)threadIdx.x < P) {
    s_pos[threadIdx.x] = a.pos_of_slot[threadIdx.x];
    s_wt[threadIdx.x] = a.pre_weighted ? 1.0f : a.pairs[2 * threadIdx.x + 1];
  }
  if (a.pairs_out && blockIdx.x == 0 && (int)threadIdx.x < P)
    a.pairs_out[threadIdx.x] = reinterpret_cast<const float2*>(a.pairs)[threadIdx.x];

  constexpr int kScWords = NS <= 4 ? 1 : NS <= 8 ? 2 : 4;
  typedef uint32_t ScaleWords __attribute__((ext_vector_type(kScWords)));
  using ScaleCell = std::conditional_t<NS == 2, uint16_t, ScaleWords>;
  struct WSet {
    u32x4 q[ND][NT];
    ScaleWords sc[NT];
    float b[NT];
    int base, count;
  };
  const uint32_t qoff = (uint32_t)((g * 16 + n) * 16);
  auto tile_of = [&](int m) { return min(tile0 + m, a.ntile - 1); };
  auto load_step = [&](WSet& ws, __amdgpu_buffer_rsrc_t rsrc, int s) {
    const uint32_t step = 4 * (wv + 4 * s) >= nblk ? 0u : (uint32_t)(wv + 4 * s) * 1024u;  // (wholly past K: zeros are contracted)
#pragma unroll
    for (int m = 0; m < NT; ++m)
      ws.q[s % ND][m] = __builtin_amdgcn_raw_buffer_load_b128(rsrc, qoff, (uint32_t)tile_of(m) * (uint32_t)nblk * 256u + step, 0);
  };
  auto plane = [&](int v) { return stream_plane_rsrc(a.groups[v].w.q_down); };
  auto load_group = [&](WSet& ws, int v) {
    const StreamGroup* gr = a.groups + v;
    const CSK_GLOBAL ScaleCell* sp = as_global(reinterpret_cast<const ScaleCell*>(gr->w.s_down)) + wv * 64 + lane;
    const CSK_GLOBAL float* bp = as_global(gr->w.b_down);
    ws.base = gr->base, ws.count = min(kStreamG, gr->left);
#pragma unroll
    for (int m = 0; m < NT; ++m) {
      const int t = tile_of(m);
      if constexpr (NS == 2) ws.sc[m][0] = sp[(size_t)t * 256];
      else ws.sc[m] = sp[(size_t)t * 256];
      ws.b[m] = bp[min(t * 16 + n, a.N - 1)];
    }
    const auto rsrc = plane(v);
#pragma unroll
    for (int s = 0; s < ND; ++s) load_step(ws, rsrc, s);
  };
  WSet ws[kSets];
#pragma unroll
  for (int i = 0; i < kSets; ++i)
    if (team + i * kMergeTeams < nvv) load_group(ws[i], team + i * kMergeTeams);

#pragma unroll 1
  for (int idx = threadIdx.x; idx < nfill; idx += kMergeThreads) {
    const int kb = idx % lrb;
    u32x4* dst = As + (size_t)idx * kMx3ChunksPerBlock;
    if (idx != (int)threadIdx.x) fetch_block(idx);
    if (kb >= nblk) {
#pragma unroll
      for (int t = 0; t < kMx3Terms; ++t) {
        dst[2 * t] = u32x4{0u, 0u, 0u, 0u};
        dst[2 * t + 1] = u32x4{0u, 0u, 127u, 0u};
      }
    } else {
      float r[32];
#pragma unroll
      for (int i = 0; i < 8; ++i) r[4 * i] = pre[i].x, r[4 * i + 1] = pre[i].y, r[4 * i + 2] = pre[i].z, r[4 * i + 3] = pre[i].w;
      mx3_quantize_terms(r, [&](int t, const u32x4& lo, const u32x4& hi) { dst[2 * t] = lo, dst[2 * t + 1] = hi; });
    }
  }
  __syncthreads();  // the rows are in LDS

  // Group v of this team out of ws, which is loaded again with group `next` (if there is one); every thread passes the barrier.
  auto group = [&](WSet& ws, int v, int next, int par) {
    float* const rbuf = red + (size_t)(par * kMergeTeams + team) * 4 * NV * 16;
    int base = 0, count = 0;
    float bias[NT];
    if (v < nvv) {
      base = ws.base, count = ws.count;
#pragma unroll
      for (int m = 0; m < NT; ++m) bias[m] = ws.b[m];
      floatx4 acc[NT];
#pragma unroll
      for (int m = 0; m < NT; ++m) acc[m] = floatx4{0.f, 0.f, 0.f, 0.f};
      int frag = ((base + min(n, count - 1)) * lrb + 4 * wv + g) * kMx3ChunksPerBlock;
      asm volatile("" : "+v"(frag));  // (fragments are read one ahead of their use, as in expert_stream_kernel)
      u32x4 flo[2], fhi[2];
      auto read_frag = [&](int i) {
        const int s = i / kMx3Terms, t = i - s * kMx3Terms;
        const u32x4* f = As + frag + (16 * s * kMx3Terms + t) * 2;
        flo[i & 1] = f[0];
        fhi[i & 1] = f[1];
      };
      read_frag(0);
      const auto rsrc = plane(v);
#pragma unroll
      for (int s = 0; s < NS; ++s) {
#pragma unroll
        for (int t = 0; t < kMx3Terms; ++t) {
          const int i = s * kMx3Terms + t;
          if (i + 1 < NS * kMx3Terms) read_frag(i + 1);
          const i32x8 aw = (i32x8)__builtin_shufflevector(flo[i & 1], fhi[i & 1], 0, 1, 2, 3, 4, 5, 6, 7);
#pragma unroll
          for (int m = 0; m < NT; ++m) {
            const int byte = (int)((ws.sc[m][s >> 2] >> (8 * (s & 3))) & 0xFFu);
            const i32x8 bw = (i32x8)__builtin_shufflevector(ws.q[s % ND][m], ws.q[s % ND][m], 0, 1, 2, 3, -1, -1, -1, -1);
            acc[m] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(aw, bw, acc[m], 2, 4, 0, aw[6], 0, byte);
          }
          // The matrix instructions stay here, where all lanes take part: the results are used by sixteen of them, and moved
          // behind that condition the instructions would read operands that only those lanes have completed, and
          // overwrite what the others still hold in the registers.
#pragma unroll
          for (int m = 0; m < NT; ++m) asm volatile("" : "+v"(acc[m]));
          __builtin_amdgcn_sched_barrier(0);
        }
        if (s + ND < NS) load_step(ws, rsrc, s + ND);
      }
      if (g == 0) {
#pragma unroll
        for (int m = 0; m < NT; ++m)
#pragma unroll
          for (int i = 0; i < 4; ++i) rbuf[(wv * NV + m * 4 + i) * 16 + n] = acc[m][i];
      }
      if (next < nvv) load_group(ws, next);
    }
    __syncthreads();
    if (v < nvv && wv == 0 && g == 0) {
#pragma unroll
      for (int m = 0; m < NT; ++m) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int o = m * 4 + i;
          const float sum = ((rbuf[(0 * NV + o) * 16 + n] + rbuf[(1 * NV + o) * 16 + n]) + rbuf[(2 * NV + o) * 16 + n]) +
                            rbuf[(3 * NV + o) * 16 + n];
          if (i < count) ys[(base + i) * (NT * 16) + m * 16 + n] = sum + bias[m];
        }
      }
    }
  };
  for (int v = 0; v < nvv; v += 2 * kMergeTeams) {  // v: the first team's; the same count of barriers in every wave
    group(ws[0], v + team, v + team + kSets * kMergeTeams, 0);
    group(ws[kSets - 1], v + team + kMergeTeams, v + team + (1 + kSets) * kMergeTeams, 1);
  }
  __syncthreads();
  for (int i = threadIdx.x; i < a.T * NT * 16; i += kMergeThreads) {
#pragma clang fp contract(off)  // w * y and the add round separately, as in the reference
    const int t = i / (NT * 16), c = i - t * (NT * 16), d = tile0 * 16 + c;
    if (d >= a.N) continue;
    float acc = 0.0f;
    for (int s = 0; s < a.k; ++s) {
      const int pos = s_pos[t * a.k + s];
      if (pos < 0) continue;  // no expert: skipped, as there
      const float y = ys[pos * (NT * 16) + c];
      if (a.pre_weighted) acc = acc + y;
      else acc = acc + s_wt[t * a.k + s] * y;
    }
    const size_t at = (size_t)t * a.N + d;
    if (a.residual) acc = a.residual[at] + acc;
    a.out[at] = acc;
  }
}

}  // namespace csk
