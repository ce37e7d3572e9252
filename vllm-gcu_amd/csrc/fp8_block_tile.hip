// 8-bit GEMMs for many rows on the MFMAs of gfx950: fp8 with 128 x 128 block scales, fp8 with per-token x per-channel
// scales (128-deep v_mfma_f32_16x16x128_f8f6f4, twice the rate of the 32-deep one), int8 with the same scales, and 16-bit
// operands (unquantised experts) on the same tiles.
//
// A workgroup owns a tile of BM = 128 .. 256 rows x 128 columns; K advances in LDS tiles of 128 bytes per row, which is exactly
// one scale block and one fp8 MFMA deep; tiles go from global memory straight into LDS (16 B per lane, no staging
// registers; 16-byte-chunk XOR swizzle, or chunk-major for kslab weights) in three stages.  Of its eight wavefronts four
// multiply -- one per SIMD with 256 registers, BM / 2 x 64 outputs each -- and four copy: a copy holds its wavefront up
// for as long as the address path is busy, 16 clocks and more each.
//
// Block scales (T8_BLOCK):
//   out[m, n] = sum_kb x_scale[m, kb] * w_scale[n / 128, kb] * sum_{k in block kb} x[m, k] * w[n, k]
// A K block's MFMA starts from zero and its result joins the running sum multiplied by the block's scale.  128 columns
// are exactly one scale block, so the weight scale of a tile and K block is a single number; it and the
// activation scales of the K block (one per row) travel with the tiles through LDS (4-byte direct-to-LDS copies).
//
// Scales outside the K sum (T8_PC, T8_INT8): every MFMA accumulates straight into the running sum, the epilogue multiplies by
// x_scale[m] (or one value) and w_scale[n] (or one value).  int8 feeds a lane's two 16-byte chunks to two 64-deep MFMAs.
//
// 16-bit operands (T8_H16: unquantised fp16 / bf16 experts at prefill token counts, grouped launches only): the tiles of 128
// bytes per row hold 64 elements; a lane's two 16-byte chunks are the operands of two 32-deep 16-bit MFMAs (chunk kq:
// elements 8 kq .. 8 kq + 7 of the first 32, chunk 4 + kq: of the second 32), which take as long as the one 128-deep fp8
// MFMA.  No scales.  The host passes K and the row strides in bytes.
//
// What bounds it: with block scales the multiply-adds (four per product of 32 clocks) beside the clock that the power limit
// leaves; else that clock alone (a K block of 256 x 128 0.86 us on the whole chip, 0.53 with operands of zeros).
#include "common.h"

#include <algorithm>
#include <cmath>
#include <type_traits>

namespace mi355q {
int kcontig_fp8_pc_launch(void* out, const void* a, const void* w, const float* a_scale, int scale_per_row,
                          const float* w_scale, int scale_per_col, const void* bias, int M, int K, int N,
                          int out_dtype, int w_layout, hipStream_t st);
bool q8_mid_call(int& rc, int mode, void* out, const void* x, const void* w, const float* x_scale, int xs_mul, const float* w_scale,
                 int ws_mul, const void* bias, int bias_f32, int M, int N, int K, long ldx, long ldo, int out_dtype, void* workspace,
                 size_t workspace_bytes, bool zeroed, hipStream_t st);
namespace {

constexpr int FTM = 256, FTN = 128, FTKB = 128;
constexpr int F8_THREADS = 512;

// operands and scales: fp8 with 128 x 128 block scales; fp8 and int8 with scales outside the K sum; 16-bit without any
enum { T8_BLOCK = 0, T8_PC = 1, T8_INT8 = 2, T8_H16 = 3 };

struct F8Args {
  void* out;                // [M, N] f16 / bf16, row stride ldo elements
  const uint8_t* x;         // [M, K] fp8, row stride ldx bytes
  const uint8_t* w;         // [N, K] fp8 row-major (row stride ldw) or in the kslab order
  const float* x_scale;     // [M, K / 128]; PC: [M] or one value
  const float* w_scale;     // [N / 128, K / 128]; PC: [N] or one value
  int xs_mul, ws_mul;       // PC, INT8: index multipliers of x_scale / w_scale (1 = per token / per channel, 0 = one value)
  int bias_f32;             // INT8: bias is f32
  const float* xs_t;        // dense launches: block scales of the activations, K block major, xs_t[kb * xs_ld + m];
  long xs_ld;               // null: x_scale as given (a row's K blocks side by side)
  const void* bias;         // [N] in the output dtype or null
  int M, N, K;
  long ldx, ldw, ldo;
  int w_kslab;              // 1: kslab order of 1-byte elements; 2: of 2-byte elements (T8_H16; K blocks of 256 bytes)
  TileOrder order;            // of the output tiles (not the grouped launches')
  int ksplits;              // > 1: every output tile is worked on by `ksplits` workgroups, each a range of K blocks,
  float* partial;           //      which leave their fp32 sums in partial[split][M][N]; the epilogue is a second launch
  // grouped (MoE) launches: a row tile is one align block of slot ids of one expert
  const int32_t* sorted_ids;   // [blocks * BM] flat (token, slot) ids, pad = numel
  const int32_t* expert_ids;   // [blocks]
  const int32_t* npp;          // device scalar: padded id count
  const float* topk_weights;   // [numel] or null
  int numel, topk, E, max_blocks;
  long w_stride, ws_stride;    // per expert: bytes of weights, floats of weight scales
};

// origin of an output tile of BM x 128 (split K: of an output tile and K range)
template <bool GROUPED, int BM>
__device__ __forceinline__ void f8_tile_origin(const F8Args& a, int mtiles, int ntiles_n, int ksplits, int tile, int& m0, int& n0, int& split) {
  int tm, tn;
  split = 0;
  if (GROUPED) {
    // block-major: neighbouring workgroups share a block's activation rows
    tm = tile / ntiles_n;
    tn = tile - tm * ntiles_n;
  } else {
    a.order.locate(tile, tm, tn, split);
  }
  m0 = tm * BM;
  n0 = tn * FTN;
}

// ---- the kernel --------------------------------------------------------------------------------------------------------
// x tiles of 16 rows pass through four register slots (six for the heights between 128 and 256, whose accumulators leave
// room); the last two x tiles of a K block are multiplied by w tile, so that each w tile is read again for the next K block
// as soon as its last product is under way, and the barrier lies before them, where the stage before has been read and the
// next one is needed.
// GROUPED: the fused-MoE grouped GEMM at prefill token counts.  Row tile b is align block b (BM slot ids of expert
// expert_ids[b]): x rows and their scales are gathered through the ids (row id / topk), weights and weight scales are the
// expert's, output row id gets the result (times its routing weight).  Blocks past num_tokens_post_pad do not exist (the
// tile count is read on the device); a block of an expert outside [0, E) writes zeros.  No K ranges, no bias.
// Against eight wavefronts that multiply and copy (us, before -> here): block scales K 7168 x N 4096 at 2048 rows 69.6 -> 60.3,
// K 8192 x N 28672 at 2048 520 -> 469; per-channel scales 409 -> 400 there; 16-bit experts 8 x (4096 x 28672) at 512 / 2048 tokens
// 514 / 1215 -> 474 / 1137, 8 x (14336 x 4096) 251 / 641 -> 227 / 632.
// x, w and, with block scales, a scale per row (1 KiB) and the tile's weight scale, 64 times
constexpr int t8_stage_bytes(int BM, int mode) { return BM * FTKB + FTN * FTKB + (mode == T8_BLOCK ? 1024 + 256 : 0); }

// scales and bias of four adjacent columns
template <int DT, int MODE>
__device__ __forceinline__ void t8_columns(const F8Args& a, int n, float* wsc, float* bias) {
  constexpr int D = DT == MI355Q_F32 ? MI355Q_F16 : DT;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    wsc[e] = MODE == T8_BLOCK || (MODE == T8_INT8 && !a.w_scale) ? 1.0f : a.w_scale[(n + e) * a.ws_mul];
    if (MODE == T8_INT8 && (DT == MI355Q_F32 || a.bias_f32)) bias[e] = a.bias ? ((const float*)a.bias)[n + e] : 0.0f;
    else bias[e] = a.bias ? Elem<D>::to_f32(((const uint16_t*)a.bias)[n + e]) : 0.0f;
  }
}
template <int MODE>
__device__ __forceinline__ float t8_row_scale(const F8Args& a, int m) {
  return MODE == T8_BLOCK || (MODE == T8_INT8 && !a.x_scale) ? 1.0f : a.x_scale[(long)m * a.xs_mul];
}

template <int DT>
__device__ __forceinline__ void t8_store4(void* out, long idx, const float* v) {
  constexpr int D = DT == MI355Q_F32 ? MI355Q_F16 : DT;
  if (DT == MI355Q_F32) {
    *(f4*)((float*)out + idx) = (f4){v[0], v[1], v[2], v[3]};
  } else {
    u2 o;
    o.x = (uint32_t)Elem<D>::from_f32(v[0]) | ((uint32_t)Elem<D>::from_f32(v[1]) << 16);
    o.y = (uint32_t)Elem<D>::from_f32(v[2]) | ((uint32_t)Elem<D>::from_f32(v[3]) << 16);
    *(u2*)((uint16_t*)out + idx) = o;
  }
}

// four adjacent outputs from their sums: scales outside the K sum, bias, rounding
template <int DT, int MODE, typename ACC>
__device__ __forceinline__ void t8_finish(const F8Args& a, long idx, const ACC& sum, float xsc, const float* wsc, const float* bias) {
  float v[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    v[e] = (float)sum[e];
    if (MODE != T8_BLOCK) v[e] = scaled_sum(v[e], xsc, wsc[e]);
    if (MODE != T8_INT8 || a.bias) v[e] = plus_bias(v[e], bias[e]);
  }
  t8_store4<DT>(a.out, idx, v);
}

template <int DT, int MODE, bool GROUPED, int BM>
__global__ void __launch_bounds__(F8_THREADS, 1)
q8_tile_kernel(F8Args a) {
  constexpr bool BLOCK = MODE == T8_BLOCK;
  typedef typename std::conditional<MODE == T8_INT8, i4, f4>::type acc_t;
  constexpr int WN = 2, NI = 4, NJ = BM / 32;           // 2 x 2 wavefronts of BM / 2 x 64 multiply, four copy
  // x tiles in registers: the first two of a K block are read while the last two of the one before are multiplied
  constexpr int XS = NJ % 4 == 0 ? 4 : 6;
  auto slot = [](int j) constexpr { return NJ % 4 == 0 || j < NJ - 2 ? j & 3 : 4 + j - (NJ - 2); };
  constexpr int X_BYTES = BM * FTKB, W_BYTES = FTN * FTKB, STAGE_BYTES = t8_stage_bytes(BM, MODE);
  constexpr int XCOPIES = BM / 8 / 4, WCOPIES = FTN / 8 / 4;       // 1 KiB copies per copying wavefront
  extern __shared__ __align__(16) unsigned char lds[];
  const int tid = threadIdx.x, lane = tid & 63, wave8 = __builtin_amdgcn_readfirstlane(tid >> 6), wave = wave8 & 3;
  const bool copies = wave8 >= 4;
  const int l16 = lane & 15, kq = lane >> 4;
  const int wm = wave / WN, wn = wave % WN;
  const int M = a.M, N = a.N, K = a.K, KB = K >> 7;

  int mtiles = (M + BM - 1) / BM;
  if (GROUPED) {
    const int blocks = (*a.npp + BM - 1) / BM;
    mtiles = __builtin_amdgcn_readfirstlane(blocks < a.max_blocks ? blocks : a.max_blocks);
  }
  const int ntiles_n = N / FTN;
  const int ksplits = (!GROUPED && a.ksplits > 1) ? a.ksplits : 1;
  const int total_tiles = mtiles * ntiles_n * ksplits;   // (split K: tile ids count (output tile, K range) pairs)
  if (GROUPED && (int)blockIdx.x >= total_tiles) return;  // (the grid is sized for the largest block count the ids can fill)
  auto tile_origin = [&](int tile, int& m0, int& n0, int& split) { f8_tile_origin<GROUPED, BM>(a, mtiles, ntiles_n, ksplits, tile, m0, n0, split); };

  const uint32_t lds_base = __builtin_amdgcn_readfirstlane((uint32_t)(size_t)(__attribute__((address_space(3))) unsigned char*)lds);
  const int nt = KB / ksplits;                     // K blocks per (output tile, K range)
  // (kept in a register: read through the dispatch packet it is fetched again in every iteration)
  const int gdim = __builtin_amdgcn_readfirstlane((int)gridDim.x);
  int tile = blockIdx.x;
  const int mytiles = (total_tiles - tile + gdim - 1) / gdim;
  const int elements = mytiles * nt;               // K blocks this workgroup multiplies, over all its tiles

  if (copies) {
    // global -> LDS: lane = 8 * row + slot, slot p of row r receives chunk p ^ (r & 7); kslab weights
    // chunk-major (lane = 8 * position + row, position p of an odd 8-row group holding chunk p ^ 1)
    const int crow = lane >> 3, cchunk = (lane & 7) ^ (crow & 7);
    uint32_t xo[XCOPIES], wo[WCOPIES], xso = 0;
    int wsbase = 0;
    const uint8_t *xtile, *wtile;
    const float* xsbase = a.x_scale;
    const long xs_kstride = (!GROUPED && a.xs_t) ? a.xs_ld : 1;       // floats between the K blocks of a row's scale
    auto set_copy_tile = [&](int tile) {
      int m0, n0, split;
      tile_origin(tile, m0, n0, split);
      long ebytes = 0;
      int escales = 0;
      if (GROUPED) {
        const int* ids = a.sorted_ids + m0;
#pragma unroll
        for (int p = 0; p < XCOPIES; ++p) {
          const int id = ids[(wave + 4 * p) * 8 + crow];
          xo[p] = (uint32_t)(max(0, min(id, a.numel - 1)) / a.topk) * (uint32_t)a.ldx + (uint32_t)(16 * cchunk);   // pads read a valid row
        }
        int e = a.expert_ids[m0 / BM];
        e = __builtin_amdgcn_readfirstlane((e < 0 || e >= a.E) ? 0 : e);     // (a foreign expert's block is computed and zeroed)
        ebytes = (long)e * a.w_stride;
        escales = e * (int)a.ws_stride;
      } else {
#pragma unroll
        for (int p = 0; p < XCOPIES; ++p) {
          const int r = (wave + 4 * p) * 8 + crow;
          xo[p] = (uint32_t)((min(m0 + r, M - 1) - m0) * a.ldx + 16 * cchunk);
        }
      }
#pragma unroll
      for (int p = 0; p < WCOPIES; ++p) {
        if (MODE == T8_H16 && a.w_kslab) {
          // 2-byte elements: a K block of the kslab order is 256 bytes per row = two of this kernel's K blocks; chunk c of
          // K block h is vector c & 3 of lane quarter 2 h + (c >> 2)
          const uint32_t n = (uint32_t)(n0 + (wave + 4 * p) * 8 + (lane & 7));
          const uint32_t c = (uint32_t)((lane >> 3) ^ (wave & 1));
          wo[p] = ((n >> 6) * (uint32_t)(K >> 8) * 4u + ((n & 63u) >> 4)) * 4096u + (c & 3u) * 1024u +
                  ((c >> 2) * 16u + (n & 15u)) * 16u;
        } else if (a.w_kslab) {
          const uint32_t n = (uint32_t)(n0 + (wave + 4 * p) * 8 + (lane & 7));
          const uint32_t c = (uint32_t)((lane >> 3) ^ (wave & 1));
          wo[p] = ((n >> 6) * (uint32_t)(K >> 7) * 4u + ((n & 63u) >> 4)) * 2048u + (c & 1u) * 1024u +
                  ((c >> 1) * 16u + (n & 15u)) * 16u;
        } else {
          const int r = (wave + 4 * p) * 8 + crow;
          wo[p] = (uint32_t)(r * a.ldw + 16 * cchunk);
        }
      }
      // activation scales: 64 rows per copying wavefront, 128-row tiles twice (32-bit index in floats from the tile's first row;
      // grouped: from the matrix's, whose scales the entry point keeps below 2^27 bytes)
      const int srow = min(64 * wave + lane, BM - 1);
      // (split K: the tile's range starts kb0 K blocks into every row; 64 kslab rows interleave their K blocks)
      const int kb0 = ksplits > 1 ? split * (KB / ksplits) : 0;
      if (!BLOCK) {
      } else if (a.xs_t && !GROUPED) {
        // K block major: the 64 scales of a copy lie side by side (4 cache lines instead of 64)
        xso = (uint32_t)(min(m0 + srow, M - 1) - m0);
        xsbase = a.xs_t + (long)kb0 * a.xs_ld + m0;
      } else if (GROUPED) {
        const int id = a.sorted_ids[m0 + srow];
        xso = (uint32_t)(max(0, min(id, a.numel - 1)) / a.topk) * (uint32_t)KB;
        xsbase = a.x_scale;
      } else {
        xso = (uint32_t)((min(m0 + srow, M - 1) - m0) * KB);
        xsbase = a.x_scale + (long)m0 * KB + kb0;
      }
      wsbase = escales + (n0 >> 7) * KB + kb0;       // the first of them copies the tile's weight scale
      xtile = GROUPED ? a.x : a.x + (long)m0 * a.ldx + (long)kb0 * FTKB;
      wtile = a.w + ebytes + (a.w_kslab ? (long)kb0 * FTKB * 64 : (long)n0 * a.ldw + (long)kb0 * FTKB);
    };
    // the K block that the next copies are of; past the last one a re-read that nobody consumes
    int kt = 0;
    set_copy_tile(tile);
    auto copy_stage = [&](int stage) {
      const uint32_t xs = lds_base + (uint32_t)(stage * STAGE_BYTES);
#pragma unroll
      for (int p = 0; p < XCOPIES; ++p) lds_copy16(xo[p], xtile + (long)kt * FTKB, xs + (uint32_t)((wave + 4 * p) * 1024));
      const long koff = MODE == T8_H16 && a.w_kslab ? (long)(kt >> 1) * 16384 + (kt & 1) * 512
                        : a.w_kslab           ? (long)kt * FTKB * 64
                                              : (long)kt * FTKB;
#pragma unroll
      for (int p = 0; p < WCOPIES; ++p) lds_copy16(wo[p], wtile + koff, xs + (uint32_t)(X_BYTES + (wave + 4 * p) * 1024));
      if (BLOCK) {
        lds_copy4(xso * 4u, xsbase + (long)kt * xs_kstride, xs + (uint32_t)(X_BYTES + W_BYTES + wave * 256));
        if (wave == 0) lds_copy4(0u, a.w_scale + wsbase + kt, xs + (uint32_t)(X_BYTES + W_BYTES + 1024));
      }
      if (++kt == nt) {
        if (tile + gdim < total_tiles) {
          tile += gdim;
          kt = 0;
          set_copy_tile(tile);
        } else {
          kt = nt - 1;
        }
      }
    };
    auto wait_all_but_last_stage = [&]() {
      constexpr int NC = XCOPIES + WCOPIES + (BLOCK ? 1 : 0);
      if (BLOCK && wave == 0) asm volatile("s_waitcnt vmcnt(%0)" : : "n"(NC + 1) : "memory");
      else asm volatile("s_waitcnt vmcnt(%0)" : : "n"(NC) : "memory");
    };
    copy_stage(0);
    copy_stage(1);
    int st = 2;
    for (int g = 0; g <= elements; ++g) {
      wait_all_but_last_stage();                   // element g has landed
      __builtin_amdgcn_s_barrier();                // ... everybody's share of it, and nobody reads element g - 1 any more
      copy_stage(st);
      st = st == 2 ? 0 : st + 1;
    }
    asm volatile("s_waitcnt vmcnt(0)" : : : "memory");   // no copy may still be writing LDS when the workgroup retires
    return;
  }

  // no row of the (only) row tile in this wavefront's share: it keeps the workgroup's barriers
  if (!GROUPED && mtiles == 1 && wm * (16 * NJ) >= M) {
    for (int g = 0; g <= elements; ++g) __builtin_amdgcn_s_barrier();
    return;
  }

  uint32_t xa[2], wa[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    xa[h] = (uint32_t)(wm * (16 * NJ) * FTKB + l16 * FTKB + (((4 * h + kq) ^ (l16 & 7)) * 16));
    wa[h] = (uint32_t)(X_BYTES + wn * (16 * NI) * FTKB) +
            (a.w_kslab ? (uint32_t)((l16 >> 3) * 1024 + (((4 * h + kq) ^ (l16 >> 3)) * 128) + (l16 & 7) * 16)
                       : (uint32_t)(l16 * FTKB + (((4 * h + kq) ^ (l16 & 7)) * 16)));
  }
  const uint32_t xsa = (uint32_t)(X_BYTES + W_BYTES) + (uint32_t)(wm * (16 * NJ) + l16) * 4u;
  struct Tile { i4 h[2]; };
  acc_t acc[NI][NJ];
  f4 ring[4];
  Tile w[NI], x[XS];
  float sc[NJ], xsn[NJ], wsn;
#pragma unroll
  for (int i = 0; i < XS; ++i) x[i].h[0] = x[i].h[1] = (i4){0, 0, 0, 0};
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    w[i].h[0] = w[i].h[1] = (i4){0, 0, 0, 0};
    ring[i] = (f4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < NJ; ++j) acc[i][j] = (acc_t){0, 0, 0, 0};
  }
#pragma unroll
  for (int j = 0; j < NJ; ++j) sc[j] = 0.f;
  auto read_x = [&](Tile& t, int j, uint32_t so) {
    t.h[0] = *(const i4*)(lds + so + xa[0] + j * 2048);
    t.h[1] = *(const i4*)(lds + so + xa[1] + j * 2048);
  };
  auto read_w = [&](Tile& t, int i, uint32_t so) {
    t.h[0] = *(const i4*)(lds + so + wa[0] + i * 2048);
    t.h[1] = *(const i4*)(lds + so + wa[1] + i * 2048);
  };
  // position p of a round: the last two x tiles of the K block before by w tile (p < 8), then the others of this one by x tile
  auto pi = [](int p) constexpr { return p < 8 ? p >> 1 : (p - 8) & 3; };
  auto pj = [](int p) constexpr { return p < 8 ? NJ - 2 + (p & 1) : (p - 8) >> 2; };
  auto add = [&](int q) {                          // the product of position q joins the running sum
    if constexpr (BLOCK) {
      acc[pi(q)][pj(q)] += sc[pj(q)] * ring[q & 3];
      // (pinned here: left alone, the compiler gives every MFMA a result tile of its own and sinks all
      // multiply-adds behind the last MFMA, where the matrix pipe waits for them)
      asm volatile("" : "+v"(acc[pi(q)][pj(q)]));
    }
  };
  auto multiply = [&](int p) {
    const int i = pi(p), j = pj(p);
    const i4 a0 = w[i].h[0], a1 = w[i].h[1], b0 = x[slot(j)].h[0], b1 = x[slot(j)].h[1];
    const i8v av = __builtin_shufflevector(a0, a1, 0, 1, 2, 3, 4, 5, 6, 7);
    const i8v bv = __builtin_shufflevector(b0, b1, 0, 1, 2, 3, 4, 5, 6, 7);
    if constexpr (BLOCK) {
      ring[p & 3] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(av, bv, (f4){0.f, 0.f, 0.f, 0.f}, 0, 0, 0, 0, 0, 0);
    } else if constexpr (MODE == T8_PC) {
      acc[i][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(av, bv, acc[i][j], 0, 0, 0, 0, 0, 0);
    } else if constexpr (MODE == T8_INT8) {
      acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a0, b0, acc[i][j], 0, 0, 0);
      acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a1, b1, acc[i][j], 0, 0, 0);
    } else if constexpr (DT == MI355Q_F16) {
      acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(bitcast<h8>(a0), bitcast<h8>(b0), acc[i][j], 0, 0, 0);
      acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(bitcast<h8>(a1), bitcast<h8>(b1), acc[i][j], 0, 0, 0);
    } else {
      acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bitcast<b8>(a0), bitcast<b8>(b0), acc[i][j], 0, 0, 0);
      acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bitcast<b8>(a1), bitcast<b8>(b1), acc[i][j], 0, 0, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  auto epilogue = [&](int tile) {
    int m0, n0, split;
    tile_origin(tile, m0, n0, split);
    // ---- epilogue: lane holds, per (w tile i, x tile j), output row m = .. + l16 and columns
    // n = .. + 4 kq + {0..3}
    if (ksplits > 1) {
      // split K: the fp32 sums of this K range, nothing else; bias (and the scales that live outside the
      // K sum) are the second launch's
      float* const part = a.partial + (long)split * M * N;
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        const int m = m0 + wm * (16 * NJ) + j * 16 + l16;
        if (m >= M) continue;
#pragma unroll
        for (int i = 0; i < NI; ++i) *(acc_t*)(part + (long)m * N + n0 + wn * (16 * NI) + i * 16 + 4 * kq) = acc[i][j];
      }
      return;
    }
    if (GROUPED) {
      const int e = a.expert_ids[m0 / BM];
      const bool foreign = e < 0 || e >= a.E;
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        const int id = a.sorted_ids[m0 + wm * (16 * NJ) + j * 16 + l16];
        if (id >= a.numel || id < 0) continue;
        const float rw = foreign ? 0.0f : (a.topk_weights ? a.topk_weights[id] : 1.0f);
#pragma unroll
        for (int i = 0; i < NI; ++i) {
          const int n = n0 + wn * (16 * NI) + i * 16 + 4 * kq;
          float v[4];
#pragma unroll
          for (int c = 0; c < 4; ++c) v[c] = foreign ? 0.0f : acc[i][j][c] * rw;
          t8_store4<DT>(a.out, (long)id * a.ldo + n, v);
        }
      }
      return;
    }
    float bia[NI][4], wsc[NI][4];
#pragma unroll
    for (int i = 0; i < NI; ++i) t8_columns<DT, MODE>(a, n0 + wn * (16 * NI) + i * 16 + 4 * kq, wsc[i], bia[i]);
    // (the scales of four row tiles requested together: loaded one by one, each waits for memory in turn)
    float xsc[4];
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const int m = m0 + wm * (16 * NJ) + j * 16 + l16;
      if (j % 4 == 0) {
#pragma unroll
        for (int k = 0; k < 4; ++k) xsc[k] = t8_row_scale<MODE>(a, min(m + 16 * k, M - 1));
      }
      if (m >= M) continue;
#pragma unroll
      for (int i = 0; i < NI; ++i) t8_finish<DT, MODE>(a, (long)m * a.ldo + n0 + wn * (16 * NI) + i * 16 + 4 * kq, acc[i][j], xsc[j % 4], wsc[i], bia[i]);
    }
  };

  int st = 0, T = 0, done = -1;                    // done: the output tile whose last K block is still being multiplied
  for (;;) {
    asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" : : : "memory");
    const uint32_t so = (uint32_t)(st * STAGE_BYTES);
    st = st == 2 ? 0 : st + 1;
#pragma unroll
    for (int p = 0; p < 8; ++p) {
      multiply(p);
      add((p + 4 * NJ - 2) % (4 * NJ));
      if (p == 0) read_x(x[slot(0)], 0, so);
      if (p == 1) read_x(x[slot(1)], 1, so);
      if (p >= 2 && (p & 1) == 0) read_w(w[(p >> 1) - 1], (p >> 1) - 1, so);
      if (p == 3 && BLOCK) {
#pragma unroll
        for (int j = 0; j < NJ; ++j) xsn[j] = *(const float*)(lds + so + xsa + j * 64);
        wsn = *(const float*)(lds + so + X_BYTES + W_BYTES + 1024);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    read_w(w[3], 3, so);
    read_x(x[slot(2)], 2, so);
    __builtin_amdgcn_sched_barrier(0);
    if (T == 0) {
      if (!BLOCK && done >= 0) epilogue(done);
      if (BLOCK && done >= 0) {
        add(6);
        add(7);
        // the two adds below find products and scales of 0: a scale of the tile before may be infinite, and Inf * 0 is NaN
        ring[2] = ring[3] = (f4){0.f, 0.f, 0.f, 0.f};
        sc[NJ - 2] = sc[NJ - 1] = 0.f;
        epilogue(done);
      }
      if (tile >= total_tiles) return;
#pragma unroll
      for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[i][j] = (acc_t){0, 0, 0, 0};
    }
    const float sa = sc[NJ - 2], sb = sc[NJ - 1];     // (positions 6 and 7 still belong to the K block before)
#pragma unroll
    for (int p = 8; p < 4 * NJ; ++p) {
      multiply(p);
      if constexpr (BLOCK) {
        if (p == 8) {
          acc[3][NJ - 2] += sa * ring[2];
#pragma unroll
          for (int j = 0; j < NJ; ++j) sc[j] = xsn[j] * wsn;
        } else if (p == 9) {
          acc[3][NJ - 1] += sb * ring[3];
        } else {
          add(p - 2);
        }
      }
      // the other x tiles of this K block, each once the tile that was in its slot is through
      if ((p & 3) == 1 && 3 + ((p - 9) >> 2) < NJ) read_x(x[slot(3 + ((p - 9) >> 2))], 3 + ((p - 9) >> 2), so);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (++T == nt) {
      T = 0;
      done = tile;
      tile += gdim;
    }
  }
}

// Second launch of a split: the ranges' sums added in range order (run-to-run identical), then the epilogue.
template <int DT, int MODE>
__global__ void __launch_bounds__(256)
q8_tile_splitk_kernel(F8Args a) {
  typedef typename std::conditional<MODE == T8_INT8, i4, f4>::type acc_t;
  const long q = (long)blockIdx.x * 256 + threadIdx.x;     // 4 adjacent columns of one row
  const int nq = a.N / 4;
  if (q >= (long)a.M * nq) return;
  const int m = (int)(q / nq), n = (int)(q % nq) * 4;
  acc_t acc = {0, 0, 0, 0};
  for (int s = 0; s < a.ksplits; ++s) acc += *(const acc_t*)(a.partial + ((long)s * a.M + m) * a.N + n);
  float wsc[4], bia[4];
  t8_columns<DT, MODE>(a, n, wsc, bia);
  t8_finish<DT, MODE>(a, (long)m * a.ldo + n, acc, t8_row_scale<MODE>(a, m), wsc, bia);
}

// Activation block scales [rows, KB] -> K block major [KB, ld] for the tile kernel's copies: a workgroup's 256
// scales of a K block then lie side by side instead of one per cache line (every column tile of a row tile reads
// them again).
__global__ void __launch_bounds__(256)
fp8_scales_kmajor_kernel(const float* xs, float* out, int rows, int KB, long ld) {
  __shared__ float t[32][33];
  const int p0 = blockIdx.x * 32, k0 = blockIdx.y * 32;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;       // 32 x 8
  for (int r = ty; r < 32; r += 8) {
    const int p = p0 + r, kb = k0 + tx;
    float v = 0.0f;
    if (p < rows && kb < KB) v = xs[(long)p * KB + kb];
    t[r][tx] = v;
  }
  __syncthreads();
  for (int r = ty; r < 32; r += 8) {
    const int kb = k0 + r, p = p0 + tx;
    if (p < rows && kb < KB) out[(long)kb * ld + p] = t[tx][r];
  }
}

int fp8_scales_kmajor_launch(const float* xs, float* out, int rows, int KB, long ld, hipStream_t st) {
  hipLaunchKernelGGL(fp8_scales_kmajor_kernel, dim3((unsigned)((rows + 31) / 32), (unsigned)((KB + 31) / 32)), dim3(256), 0, st,
                     xs, out, rows, KB, ld);
  MQ_LAUNCH_CHECK("fp8 gemm (scales, K block major)");
  return 0;
}

constexpr size_t F8_SPLITK_BYTES = (size_t)64 << 20;
constexpr size_t F8_WS_OFFSET = (size_t)1 << 20;     // the first MiB of a workspace belongs to the W4A16 arrival counters

}  // namespace

// K ranges for a shape: as many as put about one 256 x 128 tile on every CU, each at least eight K
// blocks long, a divisor of the K block count, partial sums within 64 MiB.  1: no split.
int fp8_ksplits(int M, int N, int K) {
  const long cus = device_cu_count(), tiles = (long)((M + FTM - 1) / FTM) * (N / FTN);
  const int nt = K / FTKB;
  if (N % FTN != 0 || tiles < 1 || tiles * 2 > cus) return 1;
  long s = cus / tiles;
  if (s > 8) s = 8;
  if (s > nt / 8) s = nt / 8;
  while (s > 1 && (nt % s != 0 || (size_t)s * M * N * sizeof(float) > F8_SPLITK_BYTES)) --s;
  return s < 1 ? 1 : (int)s;
}

// The height of the tiles: the cheapest by a price in us.  Rounds of workgroups (one per CU) pay a step per K block that grows
// with the height, and so does the share of the chip at work, by the power it draws; a split pays for its second launch
// and the bytes of its partial sums.  Equal tiles instead of 256 rows each and a last one that is nearly empty, and rounds
// that are full: 1537 rows are 7 x 224 on K 7168 x N 4096 (us, 256 rows -> here, block scales / per channel: 58.5 -> 56.1 / 49.8 -> 45.7), 300
// 2 x 160 on K 8192 x N 28672 (119 -> 97 / 112 -> 90), 700 4 x 192 on K 4096 x N 14336 (66 -> 60 / 62 -> 53).
// Fitted to 2000 launches for each kind of operand (25 layers, 65 .. 2048 rows, all heights, 1 .. 8 ranges), rms error 7 %; the
// pick is within 0.4 % of the best height on average, and 8 % faster than 256 rows always.
namespace {
struct T8Price {
  double base, round, step, step_bm, fill, fill_bm, split, split_mn, stream;      // stream: bytes of weights per us
};
constexpr T8Price kT8Price[3] = {{4.16, 1.65, 0.110, 0.561, 0.071, 0.266, 3.01, 1.15, 5.2e6},       // T8_BLOCK
                                 {3.86, 3.24, 0.006, 0.530, 0.161, 0.144, 1.88, 1.26, 5.2e6},       // T8_PC
                                 {4.08, 4.13, 0.065, 0.536, 0.088, 0.150, 1.12, 1.22, 5.2e6}};      // T8_INT8
}  // namespace

double t8_price(int mode, int M, int N, int K, int splits, int* height) {
  const T8Price& p = kT8Price[mode];
  const int cus = std::max(8, device_cu_count() / 8 * 8);
  const double kb = (double)(K / FTKB) / splits, stream = (double)K * N / p.stream;
  double best = 1e30;
  for (int bm = 128; bm <= 256; bm += 32) {
    const long tiles = (long)((M + bm - 1) / bm) * (N / FTN) * splits, rounds = (tiles + cus - 1) / cus;
    const double h = bm / 256.0, t = rounds * (p.round + kb * (p.step + p.step_bm * h)) + kb * tiles / cus * (p.fill + p.fill_bm * h);
    if (t < best) {
      best = t;
      if (height) *height = bm;
    }
  }
  best += p.base + (splits > 1 ? p.split + p.split_mn * 1e-6 * splits * M * N : 0);
  return std::sqrt(std::sqrt(best * best * best * best + stream * stream * stream * stream));       // (never faster than the weights arrive)
}

namespace {

template <int DT, int MODE>
int launch_f8(const F8Args& a, hipStream_t st);

template <int DT, int MODE>
int launch_f8_splitk(const F8Args& a, int splits, void* workspace, hipStream_t st) {
  F8Args b = a;
  b.ksplits = splits;
  b.partial = (float*)((char*)workspace + F8_WS_OFFSET);
  if (int rc = launch_f8<DT, MODE>(b, st)) return rc;
  const long quads = (long)a.M * (a.N / 4);
  hipLaunchKernelGGL((q8_tile_splitk_kernel<DT, MODE>), dim3((unsigned)((quads + 255) / 256)), dim3(256), 0, st, b);
  MQ_LAUNCH_CHECK("fp8 gemm (split-K epilogue)");
  return 0;
}

// Rows from which the tile kernel with K ranges side by side is ahead of the weight-streaming kernel,
// whose time grows with the rows (in steps at 17 and 33: its row tiles) while the split tile kernel's
// hardly does (measured, us at 16 / 24 / 32 / 40 / 64 rows, streaming against split: K 28672 N 8192
// 43/53/60/72/92 against 53/52/53/53/54; K 16384 N 7168 24/31/31/39/53 against 34/32/32/32/34; K 14336
// N 4096 17/21/25/32/45 against 20/21/21/21/23; K 7168 N 4096 9/12/14/18/25 against 16/16/17/17/18;
// K 8192 N 8192 14/18/19/23/30 against 23/23/22/23/24; K 8192 N 10240, three ranges, 23/29/33/42/55 against
// 31/31/31/32/33; K 4096 N 4096 7/9/10/13/16 against 15/15/15/16/17).
int fp8_split_min_rows(int N, int K, int splits) {
  (void)N;
  if (splits < 3) return 64;
  if (K >= 12288) return 24;
  if (K >= 7168) return 32;
  return 64;
}

// bytes of the K block major copy of the activation scales (rows padded to whole 64-byte lines)
size_t fp8_scales_kmajor_bytes(long rows, int K) { return (size_t)((rows + 15) / 16 * 16) * (K / FTKB) * sizeof(float); }

// with a workspace that holds the plan's partial sums: K ranges side by side; else the plain launch
template <int DT, int MODE>
int launch_f8_auto(F8Args& a, void* workspace, size_t workspace_bytes, hipStream_t st) {
  a.ksplits = 1;
  a.partial = nullptr;
  a.xs_t = nullptr;
  a.xs_ld = 0;
  const int splits = fp8_ksplits(a.M, a.N, a.K);
  const bool split = splits > 1 && workspace && workspace_bytes >= F8_WS_OFFSET + (size_t)splits * a.M * a.N * sizeof(float);
  // (It pays where a row has more scales than the one cache line that 16 K blocks share and enough tiles read them again: a launch of 4 us
  // against 0.1 us for a K block of a full round, 0.2 where all columns read the scales of one row tile.  Measured, us, as they
  // come -> K block major: K 8192 x N 17664 at 100 / 250 rows 47.9 / 69.1 -> 44.9 / 59.3, K 8192 x N 28672 at 130 / 2048 59.5 / 492 -> 53.8 / 449, K 7168
  // x N 4096 at 1537 55.8 -> 52.5, K 10368 x N 12288 at 193 56.4 -> 50.6; but K 6272 x N 10240 at 300 34.3 -> 36.1, K 7296 x N 7168 at 520
  // 42.6 -> 45.9, K 4096 x N 28672 at 80 / 130 28.8 / 33.1 -> 30.8 / 33.4, K 2048 x N 7168 at 1537 / 2048 34.5 / 40.9 -> 37.3 / 43.8.  By this rule the
  // launches of 20 layers at 80 .. 2048 rows are within 0.3 % of the better way, by the product of K blocks and tiles alone 1.5 %, 17 % at worst.)
  const long tiles = (long)((a.M + FTM - 1) / FTM) * (a.N / FTN);
  const int KB = a.K / FTKB;
  if (MODE == T8_BLOCK && workspace && ((a.M <= FTM && tiles >= 80 && KB / (split ? splits : 1) >= 40) || (KB >= 24 && KB * tiles >= 11000))) {
    // block scales: with room behind the partial sums, the activation scales are re-ordered K block major first
    const size_t off = F8_WS_OFFSET + (split ? (size_t)splits * a.M * a.N * sizeof(float) : 0);
    if (workspace_bytes >= off + fp8_scales_kmajor_bytes(a.M, a.K)) {
      float* xt = (float*)((char*)workspace + off);
      const long ld = (a.M + 15) / 16 * 16;
      if (int rc = fp8_scales_kmajor_launch(a.x_scale, xt, a.M, a.K / FTKB, ld, st)) return rc;
      a.xs_t = xt;
      a.xs_ld = ld;
    }
  }
  if (split) return launch_f8_splitk<DT, MODE>(a, splits, workspace, st);
  return launch_f8<DT, MODE>(a, st);
}

template <int DT, int MODE, int BM, bool GROUPED = false>
int launch_t8(const F8Args& a, int grid, hipStream_t st) {
  const size_t shmem = 3 * (size_t)t8_stage_bytes(BM, MODE);
  static hipError_t attr = hipFuncSetAttribute((const void*)q8_tile_kernel<DT, MODE, GROUPED, BM>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)shmem);
  MQ_REQUIRE(attr == hipSuccess, "8-bit tile gemm: cannot reserve %zu bytes of LDS: %s", shmem, hipGetErrorString(attr));
  hipLaunchKernelGGL((q8_tile_kernel<DT, MODE, GROUPED, BM>), dim3((unsigned)grid), dim3(F8_THREADS), shmem, st, a);
  MQ_LAUNCH_CHECK("8-bit tile gemm");
  return 0;
}

// The order of the tiles, measured (us, block scales / per channel / int8, tiles dealt out in turn or eight row tiles at a time where
// the columns were a multiple of eight -> here): K 9856 x N 2560 at 1300 rows 51.3 / 48.6 / 50.4 -> 43.6 / 34.3 / 37.4, at 2048
// 65.9 / 58.0 / 59.4 -> 58.7 / 47.0 / 49.2; K 3584 x N 4608 at 1537 32.5 / 30.5 / 32.0 -> 30.0 / 25.8 / 27.8; K 14336 x N 4096 at 520, two K
// ranges, 52.8 / 48.8 / 49.5 -> 47.7 / 41.9 / 43.6; K 5120 x N 13824 at 1300 108 / 106 / 109 -> 102 / 92 / 95; K 8192 x N 28672 at 2048
// 438 / 381 / 376 -> 434 / 378 / 373.
template <int DT, int MODE>
int launch_f8(const F8Args& a, hipStream_t st) {
  const int ks = a.ksplits > 1 ? a.ksplits : 1;
  int bm = 256;
  t8_price(MODE, a.M, a.N, a.K, ks, &bm);
  const int mtiles = (a.M + bm - 1) / bm, ntiles = a.N / FTN;
  F8Args b = a;
  b.order = tile_order(mtiles, ntiles, ks, (double)bm * a.K / ks, (double)FTN * a.K / ks);
  int grid = mtiles * ntiles * ks, cus = device_cu_count() / 8 * 8;
  if (cus >= 8 && grid > cus) grid = cus;
  switch (bm) {
    case 128: return launch_t8<DT, MODE, 128>(b, grid, st);
    case 160: return launch_t8<DT, MODE, 160>(b, grid, st);
    case 192: return launch_t8<DT, MODE, 192>(b, grid, st);
    case 224: return launch_t8<DT, MODE, 224>(b, grid, st);
    default: return launch_t8<DT, MODE, 256>(b, grid, st);
  }
}

// grouped launches: as many workgroups as CUs at most (the number of filled blocks is read on the device)
int f8_grouped_grid(const F8Args& a) { return (int)std::min<long>((long)a.max_blocks * (a.N / FTN), device_cu_count()); }

}  // namespace

// int8 x int8 with scales outside the K sum (null: 1): the same tiles.  Shapes and strides checked by the caller; N % 128 == 0.
int int8_tile_launch(void* out, const void* x, const void* w, const float* x_scale, int xs_mul, const float* w_scale, int ws_mul,
                     const void* bias, int bias_f32, int M, int N, int K, long ldx, long ldw, long ldo, int out_dtype,
                     void* workspace, size_t workspace_bytes, hipStream_t st) {
  F8Args a = {};
  a.out = out; a.x = (const uint8_t*)x; a.w = (const uint8_t*)w; a.x_scale = x_scale; a.w_scale = w_scale;
  a.bias = bias; a.M = M; a.N = N; a.K = K; a.ldx = ldx; a.ldw = ldw; a.ldo = ldo;
  a.w_kslab = ldw == 0 ? 1 : 0;
  a.xs_mul = xs_mul; a.ws_mul = ws_mul; a.bias_f32 = bias_f32;
  if (out_dtype == MI355Q_F16) return launch_f8_auto<MI355Q_F16, T8_INT8>(a, workspace, workspace_bytes, st);
  if (out_dtype == MI355Q_BF16) return launch_f8_auto<MI355Q_BF16, T8_INT8>(a, workspace, workspace_bytes, st);
  return launch_f8_auto<MI355Q_F32, T8_INT8>(a, workspace, workspace_bytes, st);
}

// The fused-MoE grouped GEMM with 128 x 128 block scales on align blocks of 256 or 128 slot ids: the MFMA
// tile kernel above with its rows gathered through the ids (prefill token counts; smaller blocks take the
// weight-streaming kernel).  Arguments as mi355q_moe_gemm's; checked by the caller.
int fp8_block_grouped_launch(void* out, const void* a, const void* w, const float* a_scale, const float* w_scale,
                             const float* topk_weights, const int32_t* sorted_ids, const int32_t* expert_ids,
                             const int32_t* npp, int numel, int topk, int block_size, int max_blocks, int E, int K, int N,
                             int out_dtype, int w_kslab, hipStream_t st) {
  MQ_REQUIRE(N % 128 == 0 && K % 128 == 0, "moe_gemm(fp8 tiles): N=%d and K=%d must be multiples of 128", N, K);
  MQ_REQUIRE(block_size == 256 || block_size == 128, "moe_gemm(fp8 tiles): block_size=%d must be 128 or 256", block_size);
  MQ_REQUIRE(out_dtype == MI355Q_F16 || out_dtype == MI355Q_BF16, "moe_gemm(fp8 tiles): output dtype %d", out_dtype);
  MQ_REQUIRE(((size_t)numel / topk + 1) * K < ((size_t)1 << 32) && (size_t)N * K < ((size_t)1 << 32),
             "moe_gemm(fp8 tiles): activations and one expert's weights must each stay below 4 GiB");
  F8Args g = {};
  g.out = out; g.x = (const uint8_t*)a; g.w = (const uint8_t*)w; g.x_scale = a_scale; g.w_scale = w_scale;
  g.M = numel; g.N = N; g.K = K; g.ldx = K; g.ldw = K; g.ldo = N;
  g.w_kslab = w_kslab;
  g.ksplits = 1;
  g.sorted_ids = sorted_ids; g.expert_ids = expert_ids; g.npp = npp; g.topk_weights = topk_weights;
  g.numel = numel; g.topk = topk; g.E = E; g.max_blocks = max_blocks;
  g.w_stride = (long)N * K;
  g.ws_stride = (long)(N / 128) * (K / 128);
  const int grid = f8_grouped_grid(g);
  if (block_size == 128)
    return out_dtype == MI355Q_F16 ? launch_t8<MI355Q_F16, T8_BLOCK, 128, true>(g, grid, st) : launch_t8<MI355Q_BF16, T8_BLOCK, 128, true>(g, grid, st);
  return out_dtype == MI355Q_F16 ? launch_t8<MI355Q_F16, T8_BLOCK, 256, true>(g, grid, st) : launch_t8<MI355Q_BF16, T8_BLOCK, 256, true>(g, grid, st);
}

// The same for unquantised fp16 / bf16 experts ([E, N, K] row-major, or the kslab order of 2-byte elements):
// out[id] = x[id / topk] . w[e]^T (times the routing weight), fp32 sums.
int half_grouped_tile_launch(void* out, const void* a, const void* w, const float* topk_weights,
                             const int32_t* sorted_ids, const int32_t* expert_ids, const int32_t* npp, int numel, int topk,
                             int block_size, int max_blocks, int E, int K, int N, int dtype, int w_kslab, hipStream_t st) {
  MQ_REQUIRE(N % 128 == 0 && K % 128 == 0, "moe_gemm(16-bit tiles): N=%d and K=%d must be multiples of 128", N, K);
  MQ_REQUIRE(block_size == 256 || block_size == 128, "moe_gemm(16-bit tiles): block_size=%d must be 128 or 256", block_size);
  MQ_REQUIRE(dtype == MI355Q_F16 || dtype == MI355Q_BF16, "moe_gemm(16-bit tiles): dtype %d", dtype);
  MQ_REQUIRE(((size_t)numel / topk + 1) * K * 2 < ((size_t)1 << 32) && (size_t)N * K * 2 < ((size_t)1 << 32),
             "moe_gemm(16-bit tiles): activations and one expert's weights must each stay below 4 GiB");
  F8Args g = {};
  g.out = out; g.x = (const uint8_t*)a; g.w = (const uint8_t*)w;
  g.M = numel; g.N = N; g.K = 2 * K; g.ldx = 2L * K; g.ldw = 2L * K; g.ldo = N;     // K and operand strides in bytes
  g.w_kslab = w_kslab ? 2 : 0;
  g.ksplits = 1;
  g.sorted_ids = sorted_ids; g.expert_ids = expert_ids; g.npp = npp; g.topk_weights = topk_weights;
  g.numel = numel; g.topk = topk; g.E = E; g.max_blocks = max_blocks;
  g.w_stride = 2L * N * K;
  const int grid = f8_grouped_grid(g);
  if (block_size == 128)
    return dtype == MI355Q_F16 ? launch_t8<MI355Q_F16, T8_H16, 128, true>(g, grid, st) : launch_t8<MI355Q_BF16, T8_H16, 128, true>(g, grid, st);
  return dtype == MI355Q_F16 ? launch_t8<MI355Q_F16, T8_H16, 256, true>(g, grid, st) : launch_t8<MI355Q_BF16, T8_H16, 256, true>(g, grid, st);
}

}  // namespace mi355q

using namespace mi355q;

extern "C" int mi355q_q8_tile_plan(int kind, int M, int N, int K, int* rows, int* k_ranges) {
  MQ_REQUIRE(M > 0 && N > 0 && K > 0 && N % FTN == 0 && K % FTKB == 0 && kind >= 0 && kind <= 2, "q8_tile_plan: bad shape M=%d N=%d K=%d or kind %d", M,
             N, K, kind);
  MQ_REQUIRE(rows && k_ranges, "q8_tile_plan: null pointer");
  *k_ranges = fp8_ksplits(M, N, K);
  t8_price(kind, M, N, K, *k_ranges, rows);
  return 0;
}

extern "C" size_t mi355q_fp8_gemm_workspace_bytes(int M, int N, int K) {
  if (M <= 0 || N <= 0 || K <= 0 || K % 128 != 0) return 0;
  const int s = fp8_ksplits(M, N, K);
  return s > 1 && M > fp8_split_min_rows(N, K, s) ? F8_WS_OFFSET + (size_t)s * M * N * sizeof(float) : 0;
}

extern "C" int mi355q_fp8_block_gemm(void* out, const void* x, const void* w, const float* x_scale,
                                     const float* w_scale, const void* bias, int M, int N, int K, long ldx,
                                     long ldw, long ldo, int out_dtype, void* stream) {
  return mi355q_fp8_block_gemm_ws(out, x, w, x_scale, w_scale, bias, M, N, K, ldx, ldw, ldo, out_dtype, nullptr, 0, stream);
}

extern "C" int mi355q_fp8_block_gemm_ws(void* out, const void* x, const void* w, const float* x_scale,
                                        const float* w_scale, const void* bias, int M, int N, int K, long ldx,
                                        long ldw, long ldo, int out_dtype, void* workspace, size_t workspace_bytes,
                                        void* stream) {
  const int zeroed = out_dtype & MI355Q_ZEROED_COUNTERS;
  out_dtype ^= zeroed;
  MQ_REQUIRE(M >= 0 && N > 0 && K > 0, "fp8_block_gemm: bad shape M=%d N=%d K=%d", M, N, K);
  if (M == 0) return 0;
  MQ_REQUIRE(out && x && w && x_scale && w_scale, "fp8_block_gemm: null pointer");
  MQ_REQUIRE(K % 128 == 0 && N % 128 == 0, "fp8_block_gemm: K=%d and N=%d must be multiples of 128", K, N);
  const bool kslab = ldw == 0;
  MQ_REQUIRE(ldx % 16 == 0 && ldx >= K && (kslab || (ldw % 16 == 0 && ldw >= K)),
             "fp8_block_gemm: operand row strides (%ld, %ld) must be >= K and multiples of 16", ldx, ldw);
  MQ_REQUIRE((size_t)N * K < ((size_t)1 << 32) && (size_t)M * (K / 128) < ((size_t)1 << 32) &&
                 (size_t)256 * (size_t)ldx < ((size_t)1 << 32) && (size_t)128 * (size_t)(kslab ? K : ldw) < ((size_t)1 << 32),
             "fp8_block_gemm: operands too large for 32-bit tile offsets (M=%d N=%d K=%d)", M, N, K);
  MQ_REQUIRE(ldo >= N && ldo % 4 == 0, "fp8_block_gemm: output row stride %ld must be >= N and a multiple of 4", ldo);
  MQ_REQUIRE(out_dtype == MI355Q_F16 || out_dtype == MI355Q_BF16, "fp8_block_gemm: bad out dtype %d", out_dtype);
  int rc = 0;
  if (kslab && q8_mid_call(rc, 0, out, x, w, x_scale, 0, w_scale, 0, bias, 0, M, N, K, ldx, ldo, out_dtype, workspace, workspace_bytes, zeroed != 0,
                           as_stream(stream)))
    return rc;
  F8Args a = {};
  a.out = out; a.x = (const uint8_t*)x; a.w = (const uint8_t*)w; a.x_scale = x_scale; a.w_scale = w_scale;
  a.bias = bias; a.M = M; a.N = N; a.K = K; a.ldx = ldx; a.ldw = ldw; a.ldo = ldo;
  a.w_kslab = kslab ? 1 : 0;
  a.xs_mul = a.ws_mul = 0;
  if (out_dtype == MI355Q_F16) return launch_f8_auto<MI355Q_F16, T8_BLOCK>(a, workspace, workspace_bytes, as_stream(stream));
  return launch_f8_auto<MI355Q_BF16, T8_BLOCK>(a, workspace, workspace_bytes, as_stream(stream));
}

// fp8 x fp8 with per-token (or one) activation scale and per-channel (or one) weight scale, fp32
// accumulation over the whole of K:  out[m, n] = (sum_k x[m, k] w[n, k]) * x_scale[m] * w_scale[n] (+ bias[n])
extern "C" int mi355q_fp8_scaled_gemm(void* out, const void* x, const void* w, const float* x_scale,
                                      int x_scale_per_row, const float* w_scale, int w_scale_per_col,
                                      const void* bias, int M, int N, int K, long ldx, long ldw, long ldo,
                                      int out_dtype, void* stream) {
  return mi355q_fp8_scaled_gemm_ws(out, x, w, x_scale, x_scale_per_row, w_scale, w_scale_per_col, bias, M, N, K, ldx, ldw,
                                   ldo, out_dtype, nullptr, 0, stream);
}

extern "C" int mi355q_fp8_scaled_gemm_ws(void* out, const void* x, const void* w, const float* x_scale,
                                         int x_scale_per_row, const float* w_scale, int w_scale_per_col,
                                         const void* bias, int M, int N, int K, long ldx, long ldw, long ldo,
                                         int out_dtype, void* workspace, size_t workspace_bytes, void* stream) {
  const int zeroed = out_dtype & MI355Q_ZEROED_COUNTERS;
  out_dtype ^= zeroed;
  MQ_REQUIRE(M >= 0 && N > 0 && K > 0, "fp8_scaled_gemm: bad shape M=%d N=%d K=%d", M, N, K);
  if (M == 0) return 0;
  MQ_REQUIRE(out && x && w && x_scale && w_scale, "fp8_scaled_gemm: null pointer");
  MQ_REQUIRE(K % 128 == 0 && N % 4 == 0, "fp8_scaled_gemm: K=%d must be a multiple of 128 and N=%d of 4", K, N);
  MQ_REQUIRE(out_dtype == MI355Q_F16 || out_dtype == MI355Q_BF16, "fp8_scaled_gemm: bad out dtype %d", out_dtype);
  const bool kslab = ldw == 0;
  MQ_REQUIRE(!kslab || N % 64 == 0, "fp8_scaled_gemm: weights in the kslab order need N=%d %% 64 == 0", N);
  MQ_REQUIRE(ldx >= K && (kslab || ldw >= K) && ldo >= N,
             "fp8_scaled_gemm: row strides (%ld, %ld, %ld) must cover K=%d / N=%d", ldx, ldw, ldo, K, N);
  int rc = 0;
  if (kslab && ldx % 16 == 0 && ldo % 4 == 0 &&
      q8_mid_call(rc, 1, out, x, w, x_scale, x_scale_per_row ? 1 : 0, w_scale, w_scale_per_col ? 1 : 0, bias, 0, M, N, K, ldx, ldo, out_dtype, workspace,
                  workspace_bytes, zeroed != 0, as_stream(stream)))
    return rc;
  // the MFMA tile kernel from 65 rows on when its 256 x 128 tiles fill a good part of the chip; below
  // (and for shapes it does not take) the weight-streaming kernel, which wants dense operands
  const long tiles = (long)((M + FTM - 1) / FTM) * (N / FTN);
  const bool tile_ok = N % 128 == 0 && ldx % 16 == 0 && (kslab || ldw % 16 == 0) && ldo % 4 == 0 &&
                       (size_t)N * K < ((size_t)1 << 32) && (size_t)256 * (size_t)ldx < ((size_t)1 << 32) &&
                       (size_t)128 * (size_t)(kslab ? K : ldw) < ((size_t)1 << 32);
  const bool stream_ok = ldx == K && (kslab || ldw == K) && ldo == N && (size_t)N * K * 2 < ((size_t)1 << 32) &&
                         (size_t)M * K * 2 < ((size_t)1 << 32);
  // (from 33 rows on layers of 128 tiles or more: the wavefronts without rows only copy there)
  // (and, with a workspace, wherever the split plan asks for one: K ranges side by side fill the chip)
  const size_t split_bytes = mi355q_fp8_gemm_workspace_bytes(M, N, K);
  const bool split_ok = tile_ok && workspace && split_bytes > 0 && workspace_bytes >= split_bytes;
  if (tile_ok && ((M > 64 && tiles >= 64) || (M > 32 && tiles >= 128) || split_ok || !stream_ok)) {
    F8Args a = {};
    a.out = out; a.x = (const uint8_t*)x; a.w = (const uint8_t*)w; a.x_scale = x_scale; a.w_scale = w_scale;
    a.bias = bias; a.M = M; a.N = N; a.K = K; a.ldx = ldx; a.ldw = ldw; a.ldo = ldo;
    a.w_kslab = kslab ? 1 : 0;
    a.xs_mul = x_scale_per_row ? 1 : 0;
    a.ws_mul = w_scale_per_col ? 1 : 0;
    if (out_dtype == MI355Q_F16) return launch_f8_auto<MI355Q_F16, T8_PC>(a, workspace, workspace_bytes, as_stream(stream));
    return launch_f8_auto<MI355Q_BF16, T8_PC>(a, workspace, workspace_bytes, as_stream(stream));
  }
  MQ_REQUIRE(stream_ok, "fp8_scaled_gemm: M=%d N=%d K=%d with row strides (%ld, %ld, %ld) fits neither kernel "
             "(dense operands, or N %% 128 == 0 with strides that are multiples of 16)", M, N, K, ldx, ldw, ldo);
  // the streaming kernel covers 64 rows (128 on narrow layers) per pass over the weights
  return kcontig_fp8_pc_launch(out, x, w, x_scale, x_scale_per_row, w_scale, w_scale_per_col, bias, M, K, N, out_dtype,
                               kslab ? 1 : 0, as_stream(stream));
}
