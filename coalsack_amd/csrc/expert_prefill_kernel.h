// Expert MLP for the compute-bound (prefill) regime on the block-scaled matrix
// instruction: v_mfma_scale_f32_32x32x64_f8f6f4 with A = activations as three
// FP6 (E2M3) terms (mx3.h) and B = the MXFP4 weights exactly as they are stored.
//
// Measured on this part with random operands: 5.6-6.2 PFLOP/s for FP6 x FP4 in
// the 32x32x64 form, against 1.9 PFLOP/s for bf16 32x32x16 (1.3 for 16x16x32);
// three FP6 terms instead of two bf16 terms therefore cost about half the matrix
// time, need no weight expansion (no conversion instruction at all), and the
// activation tile is 24 KiB per stage instead of 32.
//
// Operand ownership of the instruction (found by one-hot probing): lane l holds
// row l%32 of A (a token) or column l%32 of B (a weight row) and the 32 K values
// of block l/32 of the 64; position p of A pairs with position p of B; each lane
// passes the E8M0 scale of its own block.  A weight "column" l%32 is row l%16 of
// tile (l%32)/16 of a pair of packed 16-row tiles, and its 16-byte packed entry
// (32 nibbles in element order) is the operand.
//
// A workgroup of four waves owns 64 tokens of one expert (32 for the tail of an expert's
// token list) x (128 NG) weight rows -- gate and up rows of the same 64 NG features
// together, or 128 NG down rows -- and walks K in steps of 128 (4 blocks).  A wave owns NG
// groups of 32 weight rows (NG/2 gate groups and the NG/2 up groups of the same features)
// for all the tokens: NG x 2 accumulator tiles of 32 x 32, kept in the accumulation half
// of the register file, which they fill.  The activations are the expensive operand
// (three terms of 32 bytes per 32 values against 17 bytes of weights), so the tile is tall
// in weight rows: every activation fragment read from LDS feeds NG matrix instructions,
// and NG = 4 is what still leaves two workgroups per compute unit.
// The activation tile (64 tokens x 4 blocks x 3 terms x 32 B) goes to LDS by
// global_load_lds with a 16-byte XOR swizzle applied on the source side; weights go
// straight to registers; both are requested one step ahead (two LDS stages and register
// sets, one barrier per step), the weights of the step's second K half half a step later
// than the rest, so that no request is waited for sooner than half a step after it was
// made.  Scale bytes come four steps at a time, one 4-byte load per lane, row group and K half, from a plane in that
// order (common.h).  As one byte per step from the streaming kernel's plane they were two fifths of the kernel's vector
// memory instructions, and each line of them was fetched again every fourth step (gate/up, 300 tokens on 128 experts:
// 1.47 GB, now 1.2): us per layer, before / now, 2880 x 2880, top-4: 128 experts 300 tokens 409 / 375, 4096 947 / 884, 32
// experts 2048 tokens 424 / 406.
// Where a work unit's time goes (cycle counter per unit, 120b shape, 4096 tokens, two
// workgroups per compute unit at a shader clock of about 1.6 GHz): 67 us in all -- 10 us
// until the first step's operands have landed (descriptor chain, token rows, then the
// loads themselves, which take twice as long as on an idle memory system), 49 us in the K
// loop (2.1 us per step of 48 matrix instructions per wave: with the instruction at 32
// cycles the matrix pipe is 46 % busy when one workgroup of the compute unit is in its
// loop and the other is not, which is the case 56 % of the time), 8 us of epilogue.  One
// workgroup per compute unit reaches the same throughput as two (the clock rises to
// 1.9 GHz): the kernel is not short of occupancy.  With every weight request answered by
// the L2 (all units reading one tile pair: wrong results, timing only) gate/up takes 461
// instead of 558 us, so about a sixth of the time is the memory system behind the L2.
// The accumulators start from the bias.  The gate/up epilogue applies SwiGLU (hardware exp
// and reciprocal), stages each wave's 64 x 16 NG tile in LDS as fp32, re-quantises it
// to the three-term format the down GEMM reads, in place, and stores it in whole lines (a lane's own 96 bytes at
// a row's distance are 64 partial lines per instruction: 32 experts of 2880 x 2880, top-4, us per layer: 1000 tokens
// 270.9 -> 268.1, 2048 441.9 -> 436.9; 16 of 4096 x 6144, top-2, 1000 tokens 371.7 -> 368.1).
//
// Restates include/coalsack/nn/nn_ops/expert_mlp_node.h:651-732 with the token
// loop of :503-529 as the M dimension.
#pragma once
#include "common.h"
#include "expert_stream_kernel.h"
#include "mx3.h"

namespace csk {

typedef int i32x8 __attribute__((ext_vector_type(8)));

struct ExpertGemmMxArgs {
  const WorkDesc* desc;
  const int* mtiles;     // [2 * n]: (expert slot, first token) of each M tile
  const int* n_mtiles;
  const StreamGroup* groups;  // expert_stream_kernel_tiles: the M tiles as token groups, in place of the three above
  const int* n_groups;
  const int* list_row;   // packed position -> row of A; null: row = packed position
  const uint4* A;        // [rows][mx3_row_blocks(nblk)][6] x 16 B (mx3.h); blocks past nblk are zeros
  int nblk;              // K / 32
  int ntile;             // N / 16 weight row tiles (even: N is a multiple of 32)
  int n_ntiles;          // N tiles per M tile: ceil(ntile / (4 NG)) (MODE 0) or ceil(ntile / (8 NG))
  int N;
  int act_type;
  int two_part_units;    // from this many work units on, a die takes two parts of their sequence
  int cus_per_die;
  u32x4* act_out;        // MODE 0: [P][mx3_row_blocks(N / 32)][6] x 16 B
  float* y_out;          // MODE 1: [P][N]
};

constexpr int kGemmBM = 64;  // tokens per M tile of the dispatch kernels' tile list
constexpr int kDies = 8;     // accelerator dies (XCDs) of the part, each with a private L2

constexpr int kMxRowChunks = 4 * kMx3ChunksPerBlock;  // 24 chunks per token per step
constexpr int kMxWaves = 4;                           // waves per workgroup
constexpr int kMxNG = 4;                              // groups of 32 weight rows per wave

// Geometry that follows from NG (32-row weight groups per wave) and MS (32-token sub-tiles
// per work unit: 2 for an M tile of more than 32 tokens, 1 for the tail of an expert's list).
template <int NG, int MS>
struct MxGeom {
  static_assert(NG >= 2 && NG % 2 == 0, "a wave pairs NG/2 gate groups with NG/2 up groups");
  static_assert(MS == 1 || MS == 2, "one or two 32-token sub-tiles");
  static constexpr int kBM = 32 * MS;                                // tokens per workgroup
  static constexpr int kStageChunks = kBM * kMxRowChunks;            // 16-byte chunks per LDS stage
  static constexpr int kCopies = kStageChunks / 64 / kMxWaves;       // copy instructions per wave per step
  static constexpr int kFrags = 6 * MS;                              // activation fragments per step
  // LDS stages and register sets, one more than the steps of lead.  Units of few tokens (and the
  // low tile, whose accumulators leave the registers) wait for memory, not for the matrix cores: they ask
  // three steps ahead (with two stages more than one, 32 experts of 2880 x 2880, 70 tokens: 125.5 -> 119.5 us per layer; 128
  // of them, 150 tokens 365 -> 350).  Two or four stages: the four steps of the loop's body find theirs at compile time.
  static constexpr int kStages = NG == 2 && MS == 1 ? 4 : 2;
  // Floats per token in a wave's epilogue tile: whole 16-byte chunks, four banks further with every token, so that a lane's
  // blocks are read and written 16 bytes at a time without conflicts.  (The workgroup's stores read a token's chunks across the
  // waves' tiles, which begin at the same bank: two accesses for one, SQ_LDS_BANK_CONFLICT 3.6 % of the LDS cycles and 0.6 %
  // of all with 4096 tokens on 128 experts of 2880 x 2880.)  Rows of 16 NG + 1 floats were read and written 4 bytes at a
  // time (us per layer, 16 experts of 4096 x 6144, top-2, 600 tokens 287 -> 284, 64 of 1504 x 3072, top-4, 2000 tokens
  // 296.5 -> 294.4, 8 of 1024 x 512, top-8, 1000 tokens 62.9 -> 62.0).
  static constexpr int kEpiRow = 16 * NG + 4;
  static constexpr size_t kLdsBytes =
      (size_t)kStages * kStageChunks * 16 > (size_t)kMxWaves * kBM * kEpiRow * 4
          ? (size_t)kStages * kStageChunks * 16
          : (size_t)kMxWaves * kBM * kEpiRow * 4;
  static constexpr int tiles_per_wg(int mode) { return mode == 0 ? 4 * NG : 8 * NG; }
};

__device__ __forceinline__ const char* uniform_ptr(const char* p) {
  const uint64_t v = reinterpret_cast<uint64_t>(p);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)v);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(v >> 32));
  return reinterpret_cast<const char*>(((uint64_t)hi << 32) | lo);
}

// Descriptor of a whole weight plane as a raw buffer (no stride, no range to speak of: the
// offsets are tile arithmetic checked on the host).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t plane_rsrc(const void* p) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(uniform_ptr(reinterpret_cast<const char*>(p))), 0,
                                           0x7fffffff, 0x00020000);
}

typedef __attribute__((address_space(3))) const u32x4 lds_u32x4;

// One work unit: M tile (packed positions [base, base + mcount), tokens of the expert with weights `w`) x N tile nt.
// MS = 2 for M tiles that hold more than 32 tokens, MS = 1 for those that hold at most 32
// (the ragged end of an expert's token list), so that a tail of a few tokens costs one
// 32-token sub-tile of matrix work instead of two.
template <int MODE, int NG, int MS>
__device__ __forceinline__ void expert_gemm_mx_unit(const ExpertGemmMxArgs& a, const ExpertW& w, int base, int mcount,
                                                    int nt, unsigned char* smem) {
  using G = MxGeom<NG, MS>;
  constexpr int kCopies = G::kCopies, kStages = G::kStages, kLead = kStages - 1;
  static_assert(kStages * G::kStageChunks * 16 <= MxGeom<NG, 2>::kLdsBytes, "the launch asks for the LDS of full tiles");
  constexpr int kStageChunks = G::kStageChunks, kFrags = G::kFrags, kBM = G::kBM;
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // wave-uniform, and known to be
  const int n32 = lane & 31, kg = lane >> 5;
  const int n16 = n32 & 15, th = n32 >> 4;  // row within a packed tile, tile of the pair
  const int nblk = a.nblk;
  const int nsteps = (nblk + 3) >> 2;
  const int sgroups = step_scale_groups(nblk);

  // Group g of this wave is the pair of packed tiles (t0(g), t0(g) + 1).  Every address of
  // the main loop is a wave-uniform base (the group's plane and tile pair, advanced per step
  // on the scalar unit) plus a 32-bit per-lane byte offset that never changes and is the
  // same for every group, so the loads cost no vector instructions.  Nothing is clamped
  // along K: activation rows are padded with zero blocks to a whole number of steps, so
  // the weight blocks read past K (the next tile's, or the slack behind the last plane)
  // and the scale bytes read past K (padding, 127) are multiplied by exact zeros.
  // Groups past the last tile (ragged last N tile) re-read the last pair; their results
  // are dropped.  A wave none of whose groups exists (the ragged last N tile again: with
  // 2880 features three of its four waves) issues no matrix instructions at all and only
  // takes its part in copying the activation tile, which leaves its share of the matrix
  // pipe to the other workgroup on the compute unit.
  auto group_tile = [&](int g) {
    if (MODE == 0) return nt * (4 * NG) + wv * NG + 2 * (g % (NG / 2));
    return nt * (8 * NG) + wv * (2 * NG) + 2 * g;
  };
  const bool idle_wave = __builtin_amdgcn_readfirstlane((int)(group_tile(0) >= a.ntile)) != 0;
  // One buffer descriptor per weight plane; a group's tile pair and the K step go into the
  // scalar offset of the load, the lane's place within the pair into the vector offset.
  const auto q_rsrc0 = plane_rsrc(MODE == 0 ? w.q_gate : w.q_down);
  const auto q_rsrc1 = plane_rsrc(MODE == 0 ? w.q_up : w.q_down);
  const auto s_rsrc0 = plane_rsrc(MODE == 0 ? w.s_gate : w.s_down);
  const auto s_rsrc1 = plane_rsrc(MODE == 0 ? w.s_up : w.s_down);
  uint32_t goff_q[NG], goff_s[NG];  // byte offset of the group's tile pair in its planes
  const uint32_t splane = (uint32_t)step_scale_plane(a.ntile, nblk);
#pragma unroll
  for (int g = 0; g < NG; ++g) {
    const int tc = min(group_tile(g), a.ntile - 2);
    goff_q[g] = (uint32_t)__builtin_amdgcn_readfirstlane(tc * nblk * 256);
    goff_s[g] = splane + (uint32_t)__builtin_amdgcn_readfirstlane(tc * 256 * sgroups);
  }
  const uint32_t qoff = (uint32_t)(((th * nblk + kg) * 16 + n16) * 16);  // entry (tile th, block kg, row)
  const uint32_t soff = (uint32_t)step_scale_index(th, kg, n16, sgroups);
  const int rowblk = mx3_row_blocks(nblk);
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)smem;

  // LDS image of a stage: [token][24 chunks].  A token's chunks of one step are ordered by
  // the index 4 f + 2 kg + h -- f = 3 kc + term (kc: 64-wide half of the step), kg: which
  // 32-value block of that half, h: low / high 16 bytes of the term -- and chunk index c of
  // token tl sits at physical position (c & ~7) | ((c & 7) ^ ((tl >> 1) & 7)): the sixteen
  // lanes that read one chunk index of sixteen consecutive tokens then hit sixteen
  // different 16-byte bank groups.  Because kg and h occupy bits of their own in the index,
  // the swizzled position of every fragment is one of four per-lane addresses
  // (frag_addr[f & 1][h]) plus a constant.
  // Copy instruction c of wave wv fills chunks [(kCopies wv + c) * 64, +64) of the stage
  // (the LDS destinations of the instruction are fixed: lane order), so the swizzle and the
  // chunk order are applied on the source side: each lane fetches the chunk that belongs
  // at its position.
  uint32_t aoff[kCopies];  // byte offset of this lane's chunk at step 0 from a.A
#pragma unroll
  for (int c = 0; c < kCopies; ++c) {
    const int lin = (kCopies * wv + c) * 64 + lane;
    const int tl = lin / kMxRowChunks, pc = lin - tl * kMxRowChunks;
    const int ci = (pc & ~7) | ((pc & 7) ^ ((tl >> 1) & 7));        // chunk index 4 f + 2 kg + h
    const int f = ci >> 2, ckg = (ci >> 1) & 1, h = ci & 1;
    const int gch = ((2 * (f / 3) + ckg) * kMx3Terms + f % 3) * 2 + h;  // chunk of the row's step in memory
    const int tlc = min(tl, mcount - 1);  // tokens past the tile re-read its last one
    const int row = a.list_row ? a.list_row[base + tlc] : base + tlc;
    aoff[c] = (uint32_t)(((size_t)row * rowblk * kMx3ChunksPerBlock + gch) * 16);
  }
  uint32_t frag_addr[2][2];
#pragma unroll
  for (int fb = 0; fb < 2; ++fb)
#pragma unroll
    for (int h = 0; h < 2; ++h)
      frag_addr[fb][h] = lds0 + (uint32_t)((n32 * kMxRowChunks + (((fb << 2) | h) ^ (kg << 1) ^ ((n32 >> 1) & 7))) * 16);
  // LDS destination of copy c of this wave within a stage (wave-uniform)
  const uint32_t lds_wave = lds0 + (uint32_t)(kCopies * wv * 64 * 16);
  struct BSet {
    u32x4 q[2][NG];  // [64-wide K chunk of the step][row group]
  };
  // Scale bytes of four consecutive steps, one register for each: the matrix instruction picks its byte.  While four steps
  // are worked off those of the next four arrive.
  struct SSet {
    uint32_t w[2][NG];  // [64-wide K chunk of a step][row group]
  };
  SSet sc, sn;
  // copy c of the activation tile of step j into LDS stage `stage` (inline assembly: nothing
  // of it lives in a register; the explicit wait at the step boundary guarantees its arrival)
  auto issue_copy = [&](int c, int stage, int j) {
    const char* abase = reinterpret_cast<const char*>(a.A) + (size_t)j * (4 * kMx3ChunksPerBlock * 16);
    const uint32_t lds = lds_wave + (uint32_t)((stage * kStageChunks + c * 64) * 16);
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
                 :
                 : "v"(aoff[c]), "s"(abase), "s"(lds)
                 : "memory");
  };
  // Weights: buffer loads the compiler can see.  Loads hidden in inline assembly would
  // save its wait bookkeeping, but the register allocator moves values between register
  // files around the matrix instructions, and a register it moves while an untracked load
  // is still in flight takes stale data along (seen as rare wrong rows in ragged tiles).
  auto issue_q = [&](int kc, int g, BSet& b, int j) {
    const bool second = MODE == 0 && g >= NG / 2;  // up rows
    const uint32_t so = goff_q[g] + (uint32_t)j * 1024u + (uint32_t)kc * 512u;
    b.q[kc][g] = __builtin_amdgcn_raw_buffer_load_b128(second ? q_rsrc1 : q_rsrc0, qoff, so, 0);
  };
  auto issue_s = [&](int kc, int g, SSet& b, int grp) {  // steps 4 grp .. 4 grp + 3
    const bool second = MODE == 0 && g >= NG / 2;
    const uint32_t so = goff_s[g] + (uint32_t)(grp * 256 + kc * 128);
    b.w[kc][g] = __builtin_amdgcn_raw_buffer_load_b32(second ? s_rsrc1 : s_rsrc0, soff, so, 0);
  };
  // The loads of step j are issued in two parts, each spread over the fragments of half a
  // step: first the activation tile and the weights of the step's first K half, then the
  // weights of its second K half.  Loads retire in order, so at the step boundary only the
  // first part has to have landed -- the 2 NG loads of the second part stay in flight and are
  // waited for in the middle of the next step, which gives every load at least half a step
  // of lead (with one wait for everything at the boundary the last loads issued had none).
  constexpr int kHalf = kFrags / 2;
  constexpr int kFragBufs = 3;  // fragments are requested from LDS kFragBufs - 1 ahead of their use
  auto issue_part = [&](int part, int x, int stage, BSet& b, int j) {  // item x of a part
    if (part == 0) {
      if (x < kCopies) issue_copy(x, stage, j);
      if (x < NG) issue_q(0, x, b, j);
    } else if (x < NG) {
      issue_q(1, x, b, j);
    }
  };
  constexpr int kPart0Items = kCopies > NG ? kCopies : NG;

  constexpr int kWaitAll = (7 << 4) | (15 << 8);  // vmcnt(0)
  // MODE 0, end of the unit: the workgroup stores its part of the output rows, 2 NG blocks of each, from the waves'
  // tiles in LDS as 16-byte chunks numbered token by token: whole lines (a row and a unit's part of it are multiples of
  // 384 bytes).  Blocks of waves without rows are the zero padding of the last step.
  constexpr int kWaveChunks = NG / 2 * kMx3ChunksPerBlock, kOutChunks = kMxWaves * kWaveChunks;  // per token
  auto store_rows = [&] {
    const int out_rowblk = mx3_row_blocks(a.N >> 5), kb0 = nt * (2 * NG);
    const int waves = min(kMxWaves, (a.ntile - nt * (4 * NG) + NG - 1) / NG);  // those that have rows
    u32x4* o = a.act_out + ((size_t)base * out_rowblk + kb0) * kMx3ChunksPerBlock;
    // Three passes of the workgroup cover kTokens whole tokens: what a lane stores in the passes 3 q + r is the same chunk
    // of tokens kTokens apart.  All of them are requested from LDS before the first is stored: one after the other they were
    // twelve LDS latencies in a row, which a launch whose last round is short shows (64 experts of 2048 x 768, top-8, 1800
    // tokens 232.8 -> 230.0 us per layer, 32 of 2880 x 2880, top-4, 660 tokens 230.1 -> 225.4).
    constexpr int kTokens = 3 * 64 * kMxWaves / kOutChunks, kGroups = kBM / kTokens;
    static_assert(kTokens * kOutChunks == 3 * 64 * kMxWaves && kGroups * kTokens == kBM, "whole tokens, whole tiles");
#pragma unroll
    for (int r = 0; r < 3; ++r) {
      const int i = threadIdx.x + r * 64 * kMxWaves;
      const int tl = i / kOutChunks, c = i - tl * kOutChunks, w = c / kWaveChunks, cw = c - w * kWaveChunks;
      const u32x4* t = reinterpret_cast<const u32x4*>(smem) + ((w * kBM + tl) * G::kEpiRow) / 4 + 8 * (cw / kMx3ChunksPerBlock) +
                       cw % kMx3ChunksPerBlock;
      const bool rows = w < waves, stored = kb0 + c / kMx3ChunksPerBlock < out_rowblk;
      u32x4 v[kGroups];
#pragma unroll
      for (int q = 0; q < kGroups; ++q) v[q] = t[q * kTokens * G::kEpiRow / 4];
#pragma unroll
      for (int q = 0; q < kGroups; ++q) {
        if (!rows) v[q] = u32x4{0u, 0u, c & 1 ? 127u : 0u, 0u};
        if (stored && tl + q * kTokens < mcount) o[(uint32_t)((tl + q * kTokens) * out_rowblk * kMx3ChunksPerBlock + c)] = v[q];
      }
    }
  };
  if (idle_wave) {
    // the same sequence of copies, waits and barriers as below (two in front of the stores) without the weights and
    // the arithmetic; the stores of the workgroup's rows are shared out over all its waves, this one among them
#pragma unroll
    for (int u = 0; u < kLead; ++u)
#pragma unroll
      for (int c = 0; c < kCopies; ++c) issue_copy(c, u, min(u, nsteps - 1));
    int stage = kLead;  // of step j + kLead
    for (int j = 0; j < nsteps; ++j) {
      constexpr int kAhead = (kLead - 1) * kCopies;
      __builtin_amdgcn_s_waitcnt(kAhead | (7 << 4) | (15 << 8));
      __builtin_amdgcn_s_barrier();
#pragma unroll
      for (int c = 0; c < kCopies; ++c) issue_copy(c, stage, min(j + kLead, nsteps - 1));
      stage = stage + 1 == kStages ? 0 : stage + 1;
    }
    __builtin_amdgcn_s_waitcnt(kWaitAll);
    if (MODE == 0) {
      __syncthreads();
      __syncthreads();
      store_rows();
    }
    return;
  }

  floatx16 acc[MS][NG];  // [32-token sub-tile][row group]

  // Fragment i = (kc, term, 32-token sub-tile) of a step feeds NG matrix instructions (the
  // wave's row groups).  Fragments are requested from LDS two ahead of their use.  The loads
  // of the step being prefetched are issued a few per fragment between the matrix
  // instructions rather than in a burst at the step boundary: the texture address unit
  // takes 16 cycles per 64-lane 128-bit load, and a burst per wave would hold every wave at
  // the start of the step.
  auto compute = [&](const BSet& b, int stage, BSet& bn, int stage_n, int jn, int grp_n, auto phase_t, auto prefetch, auto scales) {
    constexpr int phase = decltype(phase_t)::value;
    u32x4 flo[kFragBufs], fhi[kFragBufs];
    auto read_frag = [&](int i) {
      const int kc = i / (3 * MS), t = (i % (3 * MS)) / MS, ms = i % MS;
      const int f = 3 * kc + t;
      const uint32_t off = (uint32_t)((stage * kStageChunks + ms * 32 * kMxRowChunks + (f >> 1) * 8) * 16);
      flo[i % kFragBufs] = *reinterpret_cast<lds_u32x4*>(frag_addr[f & 1][0] + off);
      fhi[i % kFragBufs] = *reinterpret_cast<lds_u32x4*>(frag_addr[f & 1][1] + off);
    };
#pragma unroll
    for (int i = 0; i < kFragBufs - 1; ++i) read_frag(i);
#pragma unroll
    for (int i = 0; i < kFrags; ++i) {
      const int kc = i / (3 * MS), ms = i % MS;
      if (i + kFragBufs - 1 < kFrags) read_frag(i + kFragBufs - 1);
      if constexpr (!decltype(prefetch)::value) {
        // nothing left to request
      } else {
        if constexpr (decltype(scales)::value && phase < 2)
          if (i < NG) issue_s(phase, i, sn, grp_n);
#pragma unroll
        for (int x = i % kHalf; x < (i < kHalf ? kPart0Items : NG); x += kHalf) issue_part(i / kHalf, x, stage_n, bn, jn);
      }
      __builtin_amdgcn_sched_barrier(0);
      // FP6 reads the first six registers; fhi[2] (register 6) is the term's scale byte
      i32x8 aw = (i32x8)__builtin_shufflevector(flo[i % kFragBufs], fhi[i % kFragBufs], 0, 1, 2, 3, 4, 5, 6, 7);
      // the fragment stays in ordinary vector registers: left to itself the register allocator
      // parks fragments in accumulation registers that it frees by moving parts of an
      // accumulator tile out and back around the matrix instructions
      asm volatile("" : "+v"(aw));
#pragma unroll
      for (int g = 0; g < NG; ++g) {
        // FP4 reads four registers
        const i32x8 bw = (i32x8)__builtin_shufflevector(b.q[kc][g], b.q[kc][g], 0, 1, 2, 3, -1, -1, -1, -1);
        acc[ms][g] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(aw, bw, acc[ms][g], 2, 4, 0,
                                                                     aw[6], phase, (int)sc.w[kc][g]);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  // Loads one (or three) steps ahead.  The step boundary is an explicit
  // wait + bare barrier: the first part of what this wave requested for step j (during step
  // j - kLead) has landed once at most the NG loads of the second part and what was
  // requested for later steps are still in flight,
  // and the barrier extends that to the other waves' parts of the activation tile and tells
  // that every wave is done reading the stage about to be overwritten.  (Scale bytes are not counted: where some of them
  // are in flight as well the wait is for more than it has to be.)
  constexpr int kSet = kCopies + 2 * NG;  // loads of a step, apart from scale bytes
  auto wait_for = [](auto sets) {  // all but the second part of the step's own and what was requested for `sets` later ones
    constexpr int n = NG + decltype(sets)::value * kSet;
    __builtin_amdgcn_s_waitcnt((n & 15) | (7 << 4) | (15 << 8) | ((n >> 4) << 14));
  };
  // First step: the biases (unconditional, the row clamped: what belongs to rows past N is
  // dropped), then the activation tile and the weights in the order of the steady state.  Behind
  // the operands, each under its own branch, the biases were four full waits in a row (20b shape, 2048
  // tokens: 462 -> 458 us per layer; 64 experts of 2048 x 768, 1000 tokens: 169.3 -> 166.9).
  float bias0[NG];
#pragma unroll
  for (int g = 0; g < NG; ++g) {
    const float* bias = MODE == 1 ? w.b_down : (g < NG / 2 ? w.b_gate : w.b_up);
    bias0[g] = as_global(bias)[min(group_tile(g) * 16 + n32, a.N - 1)];
  }
  BSet bs[kStages];
#pragma unroll
  for (int kc = 0; kc < 2; ++kc)
#pragma unroll
    for (int g = 0; g < NG; ++g) issue_s(kc, g, sn, 0);
#pragma unroll
  for (int u = 0; u < kLead; ++u) {
#pragma unroll
    for (int x = 0; x < kPart0Items; ++x) issue_part(0, x, u, bs[u], min(u, nsteps - 1));
#pragma unroll
    for (int x = 0; x < NG; ++x) issue_part(1, x, u, bs[u], min(u, nsteps - 1));
  }
#pragma unroll
  for (int g = 0; g < NG; ++g) asm volatile("" : "+v"(bias0[g]));  // (not loaded into the accumulators themselves: that spills)
  // The accumulators start from the bias of the lane's weight row,
  // so that the epilogue has neither a load nor an addition left to do for it.
#pragma unroll
  for (int g = 0; g < NG; ++g)
#pragma unroll
    for (int ms = 0; ms < MS; ++ms)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[ms][g][r] = bias0[g];
  // The accumulators live in the accumulation half of the register file (one use of that
  // register class is enough to make the compiler select the matrix instructions' form that
  // accumulates there and to split the wave's 256 registers 128 / 128): they fill it
  // exactly, and the 16-register tiles no longer compete with the weights and fragments for
  // aligned runs of ordinary registers, which made the allocator spill whole tiles.
#pragma unroll
  for (int ms = 0; ms < MS; ++ms)
#pragma unroll
    for (int g = 0; g < NG; ++g) asm volatile("" : "+a"(acc[ms][g]));

  {
    // `sets`: steps after this one whose loads may be in flight; `prefetch`, `scales`: whether it requests those of the
    // step kLead further on, and scale bytes of the next four steps.  Four steps to the loop's body, what is left
    // of them behind it: one loop body and one back edge (with an exit in the middle the compiler's wait-count pass loses
    // track and drains the load queue before the first fragment reads of every step), and behind it a pair and a single
    // step, each under one condition (as a case for each number of steps left the accumulators are spilled).  The last step
    // requests nothing: weights that nobody reads would be dropped by the compiler, and the waits count them.
    int j = 0;
    auto step = [&](auto phase_t, auto sets, auto prefetch, auto scales) {
      constexpr int phase = decltype(phase_t)::value, u = phase % kStages, un = (u + kLead) % kStages;
      wait_for(sets);
      __builtin_amdgcn_s_barrier();
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (phase == 0) sc = sn;
      compute(bs[u], u, bs[un], un, min(j + phase + kLead, nsteps - 1), min((j >> 2) + 1, sgroups - 1), phase_t, prefetch, scales);
      __builtin_amdgcn_sched_barrier(0);
    };
    using Yes = std::true_type;
    using No = std::false_type;
    using P0 = std::integral_constant<int, 0>;
    using P1 = std::integral_constant<int, 1>;
    using P2 = std::integral_constant<int, 2>;
    using P3 = std::integral_constant<int, 3>;
    using Ahead = std::integral_constant<int, kLead - 1>;
    for (; j + 3 < nsteps; j += 4) {
      step(P0{}, Ahead{}, Yes{}, Yes{});
      step(P1{}, Ahead{}, Yes{}, Yes{});
      step(P2{}, Ahead{}, Yes{}, Yes{});
      step(P3{}, Ahead{}, Yes{}, Yes{});
    }
    using More = std::integral_constant<bool, kLead == 1>;  // (with a longer lead all of them have been requested)
    const bool two = ((nsteps - j) & 2) != 0, one = ((nsteps - j) & 1) != 0;
    if (two) {
      step(P0{}, Ahead{}, More{}, No{});
      step(P1{}, std::integral_constant<int, kLead == 1 ? 0 : 1>{}, More{}, No{});
    }
    if constexpr (kStages == 4) {
      if (two && one) step(P2{}, P0{}, No{}, No{});
      if (!two && one) step(P0{}, P0{}, No{}, No{});
    } else if (one) {
      // the third step of four or the first: one copy of it, its scale bytes in place 0
#pragma unroll
      for (int kc = 0; kc < 2; ++kc)
#pragma unroll
        for (int g = 0; g < NG; ++g) sn.w[kc][g] = two ? sc.w[kc][g] >> 16 : sn.w[kc][g];
      step(P0{}, P0{}, No{}, No{});
    }
  }
  // the copies requested past the last step are still in flight: nothing may reuse their LDS before they land
  __builtin_amdgcn_s_waitcnt(kWaitAll);
  __builtin_amdgcn_sched_barrier(0);

  // epilogue: lane holds weight row n32 of each group; accumulator register r is token
  // (r % 4) + 8 * (r / 4) + 4 * kg of the 32-token sub-tile
  if (MODE == 0) {
    // bias + activation into this wave's LDS tile as fp32 [token][16 NG features + 4], then
    // one lane per token re-quantises 32 features at a time to the three-term format
    __syncthreads();  // the copies issued for the steps after the last have landed; all waves are past their reads
    float* tile = reinterpret_cast<float*>(smem) + (size_t)wv * kBM * G::kEpiRow;
    auto activate = [&](auto act_const) {
      constexpr int kAct = decltype(act_const)::value;
#pragma unroll
      for (int gi = 0; gi < NG / 2; ++gi) {
        const bool rv = group_tile(gi) * 16 + n32 < a.N;  // features past N belong to the zero padding of the output rows
#pragma unroll
        for (int ms = 0; ms < MS; ++ms) {
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const int tl = ms * 32 + (r & 3) + 8 * (r >> 2) + 4 * kg;
            const float v = moe_activation(acc[ms][gi][r], acc[ms][NG / 2 + gi][r], kAct);
            tile[tl * G::kEpiRow + 32 * gi + n32] = rv ? v : 0.0f;
          }
          // one pair of accumulator tiles at a time: left to itself the scheduler copies several
          // tiles out of the accumulation registers ahead of their use and spills one of them
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    };
    if (a.act_type == 0) activate(std::integral_constant<int, 0>{});
    else activate(std::integral_constant<int, 1>{});
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    // a lane re-quantises blocks of its token, all of them or with 32 tokens every second one, and puts them back where
    // their 32 values were
    u32x4* mine = reinterpret_cast<u32x4*>(tile + (lane % kBM) * G::kEpiRow);
#pragma unroll 1
    for (int bi = lane / kBM; bi < NG / 2; bi += 64 / kBM) {
      float v[32];
#pragma unroll
      for (int c = 0; c < 8; ++c) {
        const u32x4 four = mine[8 * bi + c];
#pragma unroll
        for (int d = 0; d < 4; ++d) v[4 * c + d] = __uint_as_float(four[d]);
      }
      u32x4 out[kMx3ChunksPerBlock];
      mx3_quantize_block(v, out);
#pragma unroll
      for (int c = 0; c < kMx3ChunksPerBlock; ++c) mine[8 * bi + c] = out[c];
    }
    __syncthreads();
    store_rows();
  } else {
    // The descriptor spans this unit's rows of y and no more: what belongs to tokens past the tile is out of its range and
    // dropped, and so is what belongs to rows past N, whose offset is moved there: an addition and a store per value, where a
    // comparison, a branch and a 64-bit product for each took (us per layer, 2880 x 2880, top-4) 32 experts 2048 tokens 411 /
    // now 404, 128 experts 300 tokens 365 / 359, 4096 890 / 878.  Stores past the caches (non-temporal, or written through)
    // change nothing.
    const uint32_t pitch = (uint32_t)a.N * 4u;
    const auto y_rsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<char*>(uniform_ptr(reinterpret_cast<const char*>(a.y_out + (size_t)base * (size_t)a.N))), 0,
        __builtin_amdgcn_readfirstlane((int)((uint32_t)mcount * pitch)), 0x00020000);
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      const int row = group_tile(g) * 16 + n32;
      const uint32_t at = row < a.N ? 4u * kg * pitch + 4u * (uint32_t)row : 0x80000000u;
#pragma unroll
      for (int ms = 0; ms < MS; ++ms) {
#pragma unroll
        for (int r = 0; r < 16; ++r)
          __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(acc[ms][g][r]), y_rsrc,
                                                at + (uint32_t)(ms * 32 + (r & 3) + 8 * (r >> 2)) * pitch, 0, 0);
      }
    }
  }
}

// Work unit = (M tile, N tile), numbered expert by expert (M-tile major for the down
// projection).  Workgroups are handed to the eight accelerator dies round-robin by linear id,
// and each die has its own L2: die x takes the x-th contiguous eighth of the unit sequence,
// so that the workgroups resident on one die at one time share a few activation panels and
// a few experts' weights, which then come from that L2 instead of from memory.
// From three units per place on the chip on, a die takes two sixteenths, the x-th and the x-th from the end: an eighth in
// one piece gives some dies more of the experts with many tokens than others, and the last die ended 10 % after the
// first (layer, us, one part / two: 128 experts of 2880 x 2880, 4096 tokens 967 / 950, 1000 tokens 511 / 501; 16 of
// 4096 x 6144, 2000 tokens 615 / 600).  With fewer units a part's ends, whose experts two dies share, weigh more (the same
// 16 experts, 1000 tokens 366 / 374; units of 256 rows: 128 experts, 300 tokens 404 / 410).
// The last of a die's units of 512 rows may be halves (halved_units): layer, us, whole units / so, 32 experts of 2880 x 2880, top-4,
// 512 tokens 188.6 / 184.6, 700 195.6 / 191.3, 1500 310 / 304, 2048 400 / 394; 16 of 4096 x 6144, top-2, 1000 tokens 334 / 319; 8 of
// 2880 x 2880, 1000 tokens 199.5 / 193.6; none of 26 such layers more than a per cent slower.  Halves of 256 rows in place
// of tokens gain as much, but with their code in the kernel the tall units hold 10 registers in memory and lose it again; always
// halving the last round, or half of it, is 1.7 and 0.9 % slower over the same layers.
template <int MODE, int NG>
__global__ __launch_bounds__(64 * kMxWaves, NG == 2 ? 3 : 2) void expert_gemm_mx_kernel(ExpertGemmMxArgs a) {
  extern __shared__ __align__(16) unsigned char smem[];
  const int n_units = *a.n_mtiles * a.n_ntiles;
  const int die = blockIdx.x % kDies;
  int slot = blockIdx.x / kDies;
  const bool two_parts = NG == kMxNG && n_units >= a.two_part_units;
  const int part = two_parts ? (n_units + 2 * kDies - 1) / (2 * kDies) : (n_units + kDies - 1) / kDies;
  const int n_slots = two_parts ? 2 * part : part;
  int half = -1;  // of the unit's 64 tokens: both, the first, the second
  if (NG == kMxNG) {
    const int whole = n_slots - halved_units(n_slots, a.cus_per_die);
    if (slot >= whole) {
      half = (slot - whole) & 1;
      slot = whole + (slot - whole) / 2;
    }
  }
  const int unit = slot < part ? die * part + slot : (2 * kDies - 2 - die) * part + slot;  // (the part 2 kDies - 1 - die)
  if (slot >= n_slots || unit >= n_units) return;
  const int mt = unit / a.n_ntiles;
  int nt = unit - mt * a.n_ntiles;
  const WorkDesc* wd = a.desc + a.mtiles[2 * mt];
  int m0 = a.mtiles[2 * mt + 1];
  if (MODE == 0) {
    // Within an expert's block of the sequence the gate/up units run N tile by N tile, the
    // expert's M tiles side by side: the workgroups resident together then read the same
    // weight rows at about the same time (20b shape, 2048 tokens: 525 -> 506 us per layer;
    // the down projection is no faster that way and keeps the M-tile-major order).
    const int tiles_e = (wd->Te + kGemmBM - 1) / kGemmBM;
    const int r = unit - (mt - m0 / kGemmBM) * a.n_ntiles;  // position within the expert's block
    nt = r / tiles_e;
    m0 = (r - nt * tiles_e) * kGemmBM;
  }
  int mcount = min(kGemmBM, wd->Te - m0);
  if (half == 1) m0 += 32, mcount -= 32;
  if (half >= 0) mcount = min(mcount, 32);
  if (mcount <= 0) return;
  if (mcount <= 32)
    expert_gemm_mx_unit<MODE, NG, 1>(a, wd->w, wd->base + m0, mcount, nt, smem);
  else
    expert_gemm_mx_unit<MODE, NG, 2>(a, wd->w, wd->base + m0, mcount, nt, smem);
}

// The same units of 256 weight rows over the streaming kernels' token groups of up to 64 tokens (self-contained records: two
// dependent reads in front of a unit's token rows, where list, descriptor and rows are three).  For batches of a few
// tokens per expert it waits for memory, and three workgroups per compute unit with three steps requested ahead each keep
// more of it in flight than the streaming kernel's groups of five to twelve tokens did, whose rows took most of the LDS (64
// experts of 2048 x 768, top-8, 50 tokens, 8 layers 587 -> 546 us; 32 of 2880 x 2880, top-4, 48 tokens 120 -> 107).
template <int MODE>
__global__ __launch_bounds__(64 * kMxWaves, 3) void expert_stream_kernel_tiles(ExpertGemmMxArgs a) {
  extern __shared__ __align__(16) unsigned char smem[];
  const int n_units = *a.n_groups * a.n_ntiles;
  const int part = (n_units + kDies - 1) / kDies;
  const int slot = blockIdx.x / kDies, unit = (blockIdx.x % kDies) * part + slot;
  if (slot >= part || unit >= n_units) return;
  const int v = unit / a.n_ntiles, nt = unit - v * a.n_ntiles;
  const StreamGroup* gr = a.groups + v;
  const int mcount = min(kGemmBM, gr->left);
  if (mcount <= 32)
    expert_gemm_mx_unit<MODE, 2, 1>(a, gr->w, gr->base, mcount, nt, smem);
  else
    expert_gemm_mx_unit<MODE, 2, 2>(a, gr->w, gr->base, mcount, nt, smem);
}

}  // namespace csk
