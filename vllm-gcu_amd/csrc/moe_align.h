// The alignment of fused-MoE slots, by one workgroup of ALIGN_WAVES wavefronts: slot ids sorted by expert, every expert's run padded to
// whole blocks.  For the launch of its own (moe_routing.hip) and for those that do something else beside it.
#pragma once
#include "common.h"

namespace mi355q {

constexpr int ALIGN_WAVES = 16;

template <typename IdT>
__device__ __forceinline__ void moe_align_ids(const IdT* __restrict__ topk_ids, int numel, int top, const int* valid_rows, int E, int B,
                 const int* expert_map, int* __restrict__ sorted_ids, int cap, int* __restrict__ expert_ids,
                 int nblocks_cap, int* __restrict__ npp, int* sm) {
  int* cnt = sm;                                 // [ALIGN_WAVES][E] per-wavefront counts -> bases
  int* estart = sm + ALIGN_WAVES * E;            // [E + 1] padded start of each expert
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int nvalid = valid_rows ? min(numel, max(0, *valid_rows) * top) : numel;

  for (int i = tid; i < ALIGN_WAVES * E; i += blockDim.x) cnt[i] = 0;
  for (int i = tid; i < cap; i += blockDim.x) sorted_ids[i] = numel;     // pads / unused tail
  __syncthreads();

  // each wavefront owns a contiguous, 64-aligned segment of the ids
  const int tiles = (nvalid + 63) / 64;
  const int tiles_per = (tiles + ALIGN_WAVES - 1) / ALIGN_WAVES;
  const int seg_b = min(nvalid, wv * tiles_per * 64), seg_e = min(nvalid, (wv + 1) * tiles_per * 64);
  for (int i = seg_b + lane; i < seg_e; i += 64) {
    const int e = (int)topk_ids[i];
    if (e >= 0 && e < E) atomicAdd(&cnt[wv * E + e], 1);
  }
  __syncthreads();
  // per expert: exclusive scan over wavefronts, total -> padded size
  for (int e = tid; e < E; e += blockDim.x) {
    int run = 0;
    for (int w = 0; w < ALIGN_WAVES; ++w) {
      int c = cnt[w * E + e];
      cnt[w * E + e] = run;
      run += c;
    }
    estart[e + 1] = (run + B - 1) / B * B;       // padded count, scanned below
  }
  __syncthreads();
  // exclusive scan of the padded counts by the first wavefront: each lane sums a run of
  // consecutive experts, the lane totals are scanned with shuffles
  if (wv == 0) {
    const int per = (E + 63) / 64;
    const int e0 = min(E, lane * per), e1 = min(E, e0 + per);
    int sum = 0;
    for (int e = e0; e < e1; ++e) sum += estart[e + 1];
    int incl = sum;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int up = __shfl_up(incl, o);
      if (lane >= o) incl += up;
    }
    int run = incl - sum;                          // exclusive prefix of this lane's run
    const int total = __shfl(incl, 63);
    // estart[e] must not be overwritten before the lane that reads estart[e + 1] = old count
    // of expert e has consumed it: every lane first reads its own run, then all write
    // a lane's run is at most 16 experts: the launch caps E at what 64 KiB of LDS hold (below 1024)
    int vals[16];
#pragma unroll
    for (int k = 0; k < 16; ++k) vals[k] = (e0 + k < e1) ? estart[e0 + k + 1] : 0;
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int k = 0; k < 16; ++k)
      if (e0 + k < e1) {
        estart[e0 + k] = run;
        run += vals[k];
      }
    if (lane == 63) estart[E] = total;
    if (lane == 0) *npp = total;
  }
  __syncthreads();
  // block -> expert table (unused blocks get expert 0)
  for (int b = tid; b < nblocks_cap; b += blockDim.x) expert_ids[b] = 0;
  __syncthreads();
  for (int e = tid; e < E; e += blockDim.x) {
    const int me = expert_map ? expert_map[e] : e;
    for (int b = estart[e] / B; b < estart[e + 1] / B; ++b) expert_ids[b] = me;
  }
  // stable scatter: tile by tile, rank inside the tile from ballots
  const int ebits = E > 1 ? 32 - __builtin_clz((unsigned)(E - 1)) : 0;
  for (int t0 = seg_b; t0 < seg_e; t0 += 64) {
    const int i = t0 + lane;
    int e = -1;
    if (i < seg_e) {
      e = (int)topk_ids[i];
      if (e < 0 || e >= E) e = -1;
    }
    // lanes of the tile that hold the same expert: the ballots of the id's bits, each taken as it is or
    // inverted according to the lane's own bit, intersected (no loop over the distinct experts of the tile)
    unsigned long long same = __ballot(e >= 0);
    for (int b = 0; b < ebits; ++b) {
      const bool bit = (e >> b) & 1;
      const unsigned long long set = __ballot(bit);
      same &= bit ? set : ~set;
    }
    int slot = 0, rank = 0;
    if (e >= 0) {
      rank = __popcll(same & ((1ull << lane) - 1ull));
      slot = estart[e] + cnt[wv * E + e] + rank;   // read before the lowest lane of the set bumps the count
    }
    __builtin_amdgcn_wave_barrier();
    if (e >= 0) {
      sorted_ids[slot] = i;
      if (rank == 0) cnt[wv * E + e] += __popcll(same);
    }
    __builtin_amdgcn_wave_barrier();
  }
}

inline size_t moe_align_lds(int E) { return ((size_t)ALIGN_WAVES * E + E + 1) * sizeof(int); }

}  // namespace mi355q
