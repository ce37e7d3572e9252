// What the kernels have in common that hold a few rows of 8-bit codes in LDS whole while the weights arrive (q8_decode.hip, q8_experts.hip): the order of the codes,
// the weights on their way, the products of a K block, the sums of the wavefronts.
#pragma once

#include "rows8.h"

namespace mi355q {

constexpr int FEW_RING = 8;                                  // tiles of 16 columns x one K block that a wavefront has on their way at most: a longer ring was slower

// (a barrier of LDS traffic alone: the weights stay on their way over it)
__device__ __forceinline__ void few_lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// Codes of `rows` rows in LDS, [K block][row][eight chunks of 16 bytes].  Chunk c of row r's K block lies at position (c >> 1 | (c & 1) << 2) ^ (r & 7), so that the
// sixteen rows and four lane quarters of an operand read fall on different banks
__device__ __forceinline__ uint32_t few_chunk_at(int rows, int kb, int r, int c) {
  return (uint32_t)((kb * rows + r) * 128 + (((c >> 1) | ((c & 1) << 2)) ^ (r & 7)) * 16);
}
// a row's part of a K block as lane quarter q multiplies it
struct FewOperand {
  u4 v[2];
  __device__ __forceinline__ FewOperand(const unsigned char* lds, int rows, int kb, int r, int q)
      : v{*(const u4*)(lds + few_chunk_at(rows, kb, r, 2 * q)), *(const u4*)(lds + few_chunk_at(rows, kb, r, 2 * q + 1))} {}
};

// offset of a lane's part of 16 columns from n on, kslab order, and one beyond the buffer, for columns that are not there
__device__ __forceinline__ uint32_t few_kslab_offset(int n, int KB, int lane) { return (uint32_t)((((n >> 6) * KB) * 4 + ((n >> 4) & 3)) * 2048 + lane * 16); }
constexpr uint32_t FEW_NONE = 0x80000000u;

// NI tiles of 16 columns, BPR K blocks of each on their way; kstride, vstride: bytes from a K block, and from a lane's first 16 bytes of it, to the next
template <int NI, int BPR>
struct FewWeights {
  static_assert(NI * BPR <= FEW_RING, "a longer ring was slower");
  u4 w[BPR][NI][2];
  __device__ __forceinline__ void ask(int b, rsrc_t res, const uint32_t* off, int kb, int KB, uint32_t kstride, uint32_t vstride) {
    const uint32_t none = kb < KB ? 0u : FEW_NONE;           // (past the last K block: no traffic)
    const int at = kb < KB ? kb * (int)kstride : 0;
#pragma unroll
    for (int t = 0; t < NI; ++t)
#pragma unroll
      for (int v = 0; v < 2; ++v) w[b][t][v] = bitcast<u4>(__builtin_amdgcn_raw_buffer_load_b128(res, (int)(off[t] | none), at + v * (int)vstride, 2));
  }
};
// the products of a K block, added to `part`
__device__ __forceinline__ f4 few_fp8_products(const u4* w, const FewOperand& x, f4 part) {
#pragma unroll
  for (int v = 0; v < 2; ++v) {
    const u4 wv = w[v];
    part = __builtin_amdgcn_mfma_f32_16x16x32_fp8_fp8((long)((unsigned long)wv[0] | ((unsigned long)wv[1] << 32)),
                                                      (long)((unsigned long)x.v[v][0] | ((unsigned long)x.v[v][1] << 32)), part, 0, 0, 0);
    part = __builtin_amdgcn_mfma_f32_16x16x32_fp8_fp8((long)((unsigned long)wv[2] | ((unsigned long)wv[3] << 32)),
                                                      (long)((unsigned long)x.v[v][2] | ((unsigned long)x.v[v][3] << 32)), part, 0, 0, 0);
  }
  return part;
}

// K blocks wave, wave + W, .. of the KB, the first BPR of which are on their way (ask(b, kb); KB >= 1 and wave < W)
template <int BPR, int W, typename Multiply, typename Ask>
__device__ __forceinline__ void few_walk(int KB, int wave, Multiply multiply, Ask ask) {
  const int mine = (KB - wave + W - 1) / W;
  int i = 0;
  for (; i + BPR < mine; i += BPR) {
#pragma unroll
    for (int b = 0; b < BPR; ++b) {
      multiply(b, wave + W * (i + b));
      ask(b, wave + W * (i + b + BPR));
    }
  }
#pragma unroll
  for (int b = 0; b < BPR; ++b)
    if (i + b < mine) multiply(b, wave + W * (i + b));
}

// a tile's sum over the wavefronts, in their order; sums: [wavefront][tile of `tiles`][lane]
template <int W, typename Acc>
__device__ __forceinline__ Acc few_sum(const Acc* sums, int tiles, int tile, int lane) {
  Acc sum = sums[tile * 64 + lane];
#pragma unroll
  for (int s = 1; s < W; ++s) sum += sums[(s * tiles + tile) * 64 + lane];
  return sum;
}

}  // namespace mi355q
