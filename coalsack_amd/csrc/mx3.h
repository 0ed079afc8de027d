// Activations as three block-scaled FP6 terms, the A operand of the scaled
// matrix instructions (v_mfma_scale_f32_32x32x64_f8f6f4, A = E2M3, B = E2M1).
//
// A block of 32 consecutive values x is written as
//     x = 2^(s0-127) q0 + 2^(s1-127) q1 + 2^(s2-127) q2 + r,
// q_t = 32 E2M3 codes (sign, 2 exponent bits, 3 mantissa bits; |q| <= 7.5), each
// term the round-to-nearest of what the terms before it left over, its scale
// chosen so that the largest leftover lands in [4, 8).  Every term removes at
// least 4.9 bits of the block maximum, so |r| <= 2^-14.7 max|x| and, measured on
// N(0,1) rows, a 2880-long contraction differs from fp32 by 2.3e-5 relative rms.
// The MXFP4 weights are the instruction's B operand as they are stored (codes and
// E8M0 scale bytes are the hardware's own), products are exact, sums are fp32.
//
// Storage: [row][K/32][3 terms] x 32 bytes:
//     bytes 0..23  32 codes x 6 bits, code j at bits [6j, 6j+6) (little endian)
//     byte  24     E8M0 scale byte of the term
//     bytes 25..31 zero
// so a lane's operand for one matrix instruction is two aligned 16-byte chunks
// and carries its own scale.
#pragma once
#include "common.h"

namespace csk {

constexpr int kMx3Terms = 3;
constexpr int kMx3ChunksPerBlock = 2 * kMx3Terms;  // 16-byte chunks per 32-value block

// Rows are padded with all-zero blocks (codes 0, scale byte 127) to a whole number of the
// GEMM's four-block K steps, so that the GEMM never has to clamp or mask at the end of K.
__host__ __device__ inline int mx3_row_blocks(int nblk) { return (nblk + 3) & ~3; }

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x32 __attribute__((ext_vector_type(32)));
typedef uint32_t u32x6 __attribute__((ext_vector_type(6)));

// Quantises one block held in registers; put(t, lo, hi) takes the two chunks of term t.
// v_cvt_scalef32_2xpk16_fp6_f32 divides by the scale, rounds to nearest even, saturates
// at +-7.5 and packs value i of its first operand at position 2i, of its second at
// 2i+1; v_cvt_scalef32_pk32_f32_fp6 is its inverse in position order (both probed).
template <class Put>
__device__ __forceinline__ void mx3_quantize_terms(float (&r)[32], Put put) {
#pragma unroll
  for (int t = 0; t < kMx3Terms; ++t) {
    uint32_t eb;
    if (t == 0) {
      // the maximum of the magnitudes as integers: unlike a floating-point maximum it keeps a
      // NaN (and an infinity), which then shows as exponent byte 255
      uint32_t mb = 0u;
#pragma unroll
      for (int j = 0; j < 32; ++j) mb = max(mb, __float_as_uint(r[j]) & 0x7fffffffu);
      eb = mb >> 23;
    } else {
      float m = 0.0f;
#pragma unroll
      for (int j = 0; j < 32; ++j) m = fmaxf(m, fabsf(r[j]));
      eb = (__float_as_uint(m) >> 23) & 0xffu;
    }
    // block maximum / scale in [4, 8); blocks below 2^-124 are stored as zeros.  A block
    // that holds a NaN or an infinity gets scale byte 255 on its first term -- the E8M0 NaN,
    // which the matrix instruction turns into NaN products: every output of that row is then
    // NaN, as in fp32 arithmetic, instead of a saturated finite value.
    const bool nonfinite = t == 0 && eb == 255u;
    const uint32_t s = nonfinite ? 255u : eb < 3u ? 127u : min(eb - 2u, 252u);
    const float sc = __uint_as_float(min(s, 252u) << 23);  // 2^(s-127)
    f32x16 ev, od;
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      ev[j] = r[2 * j];
      od[j] = r[2 * j + 1];
    }
    u32x6 q = __builtin_amdgcn_cvt_scalef32_2xpk16_fp6_f32(ev, od, sc);
    // The conversion takes several passes and writes its first results before it has read its
    // last operands, which the compiler does not know: with the result placed over part of
    // the operands (seen at an offset of two registers) the term comes out wrong.  Keeping the
    // operands alive past it keeps the registers apart.
    asm volatile("" : "+v"(q) : "v"(ev), "v"(od), "v"(sc));
    if (t + 1 < kMx3Terms) {
      f32x32 d = __builtin_amdgcn_cvt_scalef32_pk32_f32_fp6(q, sc);
      asm volatile("" : "+v"(d) : "v"(q), "v"(sc));  // (this one, too, writes 32 registers over several passes)
#pragma unroll
      for (int j = 0; j < 32; ++j) r[j] = r[j] - d[j];  // exact: d is r rounded to 4 bits
    }
    put(t, u32x4{q[0], q[1], q[2], q[3]}, u32x4{q[4], q[5], s, 0u});
  }
}
// out[2t], out[2t+1] are the chunks of term t.
__device__ __forceinline__ void mx3_quantize_block(float (&r)[32], u32x4 (&out)[kMx3ChunksPerBlock]) {
  mx3_quantize_terms(r, [&](int t, const u32x4& lo, const u32x4& hi) { out[2 * t] = lo, out[2 * t + 1] = hi; });
}

// rows of fp32 -> three-term FP6 blocks, one thread per block (padding blocks included):
//   x3[(row * mx3_row_blocks(nblk) + kb) * 6 + c] <- quantise(x[src(row)][32 kb .. 32 kb + 31] * w(row))
// src(row) = gather_tok[row] and w(row) = gather_w[row] when given (rows gathered and
// pre-scaled per dispatch position, expert_mlp_node.h:515-522), else row and 1.
//
// A wave takes 64 consecutive blocks of the output.  A block is 128 bytes in and 96 out, so a
// lane that loads and stores its own block touches 64 lines per instruction; here the wave loads 1 KiB of
// consecutive input per instruction, turns it in LDS, and stores 1 KiB of consecutive output.
// As riders of the top-k launch (2048 tokens of 2880: 31.4 -> 27.4 us, 4096: 40.9 -> 37.3) what is left
// is the top-k kernel's own longest workgroup; layer of 64 experts, 2048 x 768, 1000 tokens 172.5 -> 170.
constexpr int kMx3Pitch = 36;  // floats per block in LDS: 16-byte aligned, and the lanes' blocks start in different banks
constexpr int kMx3LdsWave = 64 * kMx3Pitch;  // floats per wave
__device__ __forceinline__ void mx3_rows_wave(long b0, const float* __restrict__ x, u32x4* __restrict__ x3,
                                              long rows, int nblk, const int* __restrict__ gather_tok,
                                              const float* __restrict__ gather_w, float* lds) {
  const int rowblk = mx3_row_blocks(nblk);
  const long total = rows * rowblk;
  if (b0 >= total) return;
  const int lane = threadIdx.x & 63;
  float4* l4 = reinterpret_cast<float4*>(lds);
  {
    // load i of a lane is part lane % 8 of block b0 + 8 i + lane / 8
    const int part = lane & 7;
    long row = (b0 + (lane >> 3)) / rowblk;
    int kb = (int)((b0 + (lane >> 3)) - row * rowblk);
    float4 v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      v[i] = make_float4(0.f, 0.f, 0.f, 0.f);
      if (row < rows && kb < nblk) {
        const long srow = gather_tok ? gather_tok[row] : row;
        v[i] = reinterpret_cast<const float4*>(x + (srow * nblk + kb) * 32)[part];
        if (gather_w) {
          const float gw = gather_w[row];
          v[i].x *= gw, v[i].y *= gw, v[i].z *= gw, v[i].w *= gw;
        }
      }
      kb += 8;
      while (kb >= rowblk) kb -= rowblk, ++row;
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) l4[(8 * i + (lane >> 3)) * (kMx3Pitch / 4) + part] = v[i];
  }
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  float r[32];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const float4 v = l4[lane * (kMx3Pitch / 4) + i];
    r[4 * i] = v.x, r[4 * i + 1] = v.y, r[4 * i + 2] = v.z, r[4 * i + 3] = v.w;
  }
  // (a padding block is 32 zeros: codes 0 and scale byte 127 on every term)
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  u32x4* o4 = reinterpret_cast<u32x4*>(lds);
  mx3_quantize_terms(r, [&](int t, const u32x4& lo, const u32x4& hi) {
    o4[lane * kMx3ChunksPerBlock + 2 * t] = lo;
    o4[lane * kMx3ChunksPerBlock + 2 * t + 1] = hi;
  });
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  const long n_out = min((total - b0), 64L) * kMx3ChunksPerBlock;
  u32x4* dst = x3 + b0 * kMx3ChunksPerBlock;
#pragma unroll
  for (int c = 0; c < kMx3ChunksPerBlock; ++c) {
    const int i = c * 64 + lane;
    if (i < n_out) dst[i] = o4[i];
  }
}
__global__ __launch_bounds__(256) void mx3_rows_kernel(const float* __restrict__ x,
                                                       u32x4* __restrict__ x3, long rows, int nblk,
                                                       const int* __restrict__ gather_tok,
                                                       const float* __restrict__ gather_w) {
  __shared__ __align__(16) float lds[4 * kMx3LdsWave];
  const int wv = threadIdx.x >> 6;
  mx3_rows_wave((long)blockIdx.x * 256 + wv * 64, x, x3, rows, nblk, gather_tok, gather_w, lds + wv * kMx3LdsWave);
}

// The same work as a rider of another kernel's launch: workgroups first_wg, first_wg + 1, ...
// of that kernel's grid write the rows (x3 == nullptr: no such workgroups were launched).
struct Mx3Rider {
  const float* x;
  u32x4* x3;
  long rows;
  int nblk;
  int first_wg;
};

}  // namespace csk
