// Up to 64 (token, slot) ids as one workgroup sees them without an alignment: the slots of an expert in blocks of 2^SHIFT, experts in the order of
// their first slot.  Every wavefront finds block z by itself, from ballots of the bits of the experts' numbers.
#pragma once

#include "common.h"

namespace mi355q {

struct SlotBlock {
  int expert, real;            // real: slots of the block, 0 where there is no block z
  int mine, rank, chunk;       // this lane's slot's expert (-1: none of the E), its rank among that expert's slots, and the block's number among those of its expert
};

// ids: the slots' experts, every `step`th int32; bits: of an expert's number
template <int SHIFT>
__device__ __forceinline__ SlotBlock find_slot_block(const int32_t* ids, int step, int bits, int numel, int E, int z, int lane) {
  constexpr int B = 1 << SHIFT;
  SlotBlock b;
  b.mine = lane < numel ? ids[lane * step] : -1;
  if (b.mine >= E) b.mine = -1;
  unsigned long long same = __ballot(b.mine >= 0);
  for (int i = 0; i < bits; ++i) {
    const bool bit = (b.mine >> i) & 1;
    const unsigned long long set = __ballot(bit);
    same &= bit ? set : ~set;
  }
  const unsigned long long below = (1ull << lane) - 1ull;
  const int slots = b.mine >= 0 ? __popcll(same) : 0;
  b.rank = __popcll(same & below);
  int first = 0;               // the expert's first block
#pragma unroll
  for (int n = 0; n < 64; n += B) first += __popcll(__ballot(b.rank == 0 && slots > n) & below);
  const unsigned long long found = __ballot(b.mine >= 0 && b.rank == 0 && z >= first && z < first + (slots + B - 1) / B);
  b.real = 0;
  if (!found) return b;        // (as in every wavefront of the workgroup)
  const int owner = __builtin_amdgcn_readfirstlane(__ffsll(found) - 1);
  b.expert = __builtin_amdgcn_readlane(b.mine, owner);
  b.chunk = z - __builtin_amdgcn_readlane(first, owner);
  b.real = min(B, __builtin_amdgcn_readlane(slots, owner) - B * b.chunk);
  return b;
}
// whether the block holds this lane's slot, at position rank % 2^SHIFT
template <int SHIFT>
__device__ __forceinline__ bool holds_lane(const SlotBlock& b) { return b.mine == b.expert && b.rank >> SHIFT == b.chunk; }

}  // namespace mi355q
