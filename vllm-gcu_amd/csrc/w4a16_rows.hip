// W4A16 MFMA GEMM for a few dozen to some hundred rows.
//
// Between the decode kernel (up to 16 rows, 32 on some layers) and the prefill kernels the weights are still read about
// once, so a launch is a stream of them with an LDS image of the activations beside it.  What bounds it: per K block of
// 128 a CU moves 8 KiB of weights and 256 bytes per row into LDS, and its SIMDs issue nine vector instructions per packed
// word to make operands of it; both take about as long (K 4096 x N 28672, 64 rows: 19.1 us for the copies alone, 19.5 for the
// arithmetic alone).  Everything here is about running the two side by side:
//   - wavefronts of their own copy (two per K range, one range per half of K): a copy instruction that waits for the
//     address path holds up only its wavefront (the same loop with every wavefront copying its share: 27.2 us, with the copies
//     spread between the matrix instructions 24.4, with copying wavefronts 23.5);
//   - a wavefront that computes owns NT tiles of 16 columns x all rows of the workgroup, so no weight is dequantised twice
//     in a workgroup, and A operands are read from LDS one K step ahead;
//   - K is cut inside the workgroup (KS ranges, sums meet in LDS): as many wavefronts per SIMD as two workgroups
//     give, without partial sums in memory;
//   - tiles of 32..64 rows x 64 columns, two workgroups per CU, for layers of few columns, 32..96 x 128, one per CU,
//     for wide ones.
// Everything a stage needs travels from global memory straight into LDS by instructions issued from inline assembly
// (the compiler, which does not see them, waits for the LDS reads alone); they are waited for by hand.
//
// B operands are the exact integers q - z in the activation type and the group scale multiplies the fp32 partial sum of
// each group, as in the 64-row tile kernel: the only rounding is that of the fp32 additions, for fp16 and bf16 alike.  What a
// pre-scaled zero-point holds beyond an integer times the scale is taken off behind each K block.
//
// Measured (us, fp16, groups of 128, weights cold; before -> here): 4096 x 4096 at 48 / 96 / 192 rows 12.0 / 15.5 / 23.1 ->
// 9.1 / 9.4 / 12.2; 4096 x 6144 at 64 / 128 / 256 15.9 / 20.5 / 28.2 -> 9.5 / 13.2 / 18.6; 4096 x 28672 at 48 / 64 / 96
// 29.9 / 32.7 / 41.7 -> 20.3 / 23.2 / 29.1; 14336 x 4096 at 48 / 96 / 192 20.3 / 27.5 / 39.0 -> 16.3 / 21.9 / 31.7.
// A workgroup without another one on its CU takes a ring of three stages in place of two, and the tiles up to 128 rows are priced for it (before -> since):
// 4096 x 6144 at 96 15.4 -> 11.9; 8192 x 8192 at 40 / 96 18.1 / 29.8 -> 16.1 / 21.8; 4096 x 12288 at 48 16.1 -> 12.9; 5120 x 13824 at 40 19.7 -> 15.5;
// 11008 x 4096 at 48 16.5 -> 14.3; 4096 x 28672 at 24 19.4 -> 17.1; bf16 8192 x 8192 at 48 / 96 21.2 / 29.9 -> 18.1 / 25.0.
#include "common.h"

#include <algorithm>
#include <cmath>

namespace mi355q {

int w4a16_splitk_reduce_launch(void* out, const float* partial, const void* bias, int M, int N, int splits,
                               int dtype, hipStream_t st);

namespace {

struct RowsArgs {
  uint16_t* out;
  const uint16_t* x;
  const u4* qw;
  const uint16_t* scales;
  const char* zeros;          // packed int4, or z * s in the activation type
  const uint16_t* bias;
  int M, K, N;
  int kper;                   // K blocks per range (blockIdx.y)
  uint32_t gpk_magic;         // ceil(2^32 / K blocks per group), 0: a group is one K block or less
  int mtiles;
  float* partial;             // split K: f32 tiles [range][M][N]; null: write the output
  // grouped (fused-MoE) launches: blockIdx.y = block of sorted token slots, all of one expert
  const int32_t* sorted_ids;    // slot ids, pads >= numel
  const int32_t* expert_ids;    // [blocks]
  const int32_t* npp;           // device scalar: slots after padding
  const float* topk_weights;    // [numel] or null
  int numel, topk, E, block;
  long w_stride, s_stride, z_stride;   // bytes per expert
};

struct RowsDq {
  uint32_t magic, mlo, mhi;
};
template <int DT> struct RowsMma;
template <> struct RowsMma<MI355Q_F16> {
  static __device__ __forceinline__ f4 run(const u4& a, const u4& b, f4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(bitcast<h8>(a), bitcast<h8>(b), c, 0, 0, 0);
  }
  // one packed word -> 8 values q - z; zl = 1024 + z, zh = 64 + z
  static __device__ __forceinline__ u4 dequant(uint32_t w, _Float16 zl, _Float16 zh, const RowsDq& k) {
    const h2 zlo = {zl, zl}, zhi = {zh, zh}, sixteenth = {(_Float16)0.0625f, (_Float16)0.0625f};
    const uint32_t w8 = w >> 8;
    const h2 r0 = bitcast<h2>((w & k.mlo) | k.magic) - zlo;                                          // 1024 + q
    const h2 r1 = __builtin_elementwise_fma(bitcast<h2>((w & k.mhi) | k.magic), sixteenth, -zhi);    // 1024 + 16 q
    const h2 r2 = bitcast<h2>((w8 & k.mlo) | k.magic) - zlo;
    const h2 r3 = __builtin_elementwise_fma(bitcast<h2>((w8 & k.mhi) | k.magic), sixteenth, -zhi);
    return (u4){bitcast<uint32_t>(r0), bitcast<uint32_t>(r1), bitcast<uint32_t>(r2), bitcast<uint32_t>(r3)};
  }
};
template <> struct RowsMma<MI355Q_BF16> {
  static __device__ __forceinline__ f4 run(const u4& a, const u4& b, f4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(bitcast<b8>(a), bitcast<b8>(b), c, 0, 0, 0);
  }
  // the same fp16 patterns through one mixed-precision multiply-add per weight (exact in fp32) and a packed conversion
  static __device__ __forceinline__ uint32_t pair(h2 a, float m, _Float16 z) {
    typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
    const bf2 r = {(__bf16)__builtin_fmaf((float)a.x, m, -(float)z), (__bf16)__builtin_fmaf((float)a.y, m, -(float)z)};
    return bitcast<uint32_t>(r);
  }
  static __device__ __forceinline__ u4 dequant(uint32_t w, _Float16 zl, _Float16 zh, const RowsDq& k) {
    float one = 1.0f, sixteenth = 0.0625f;
    asm volatile("" : "+s"(one));                     // (as a literal the multiplication folds away and the
    asm volatile("" : "+s"(sixteenth));               //  conversion becomes an instruction of its own)
    const uint32_t w8 = w >> 8;
    return (u4){pair(bitcast<h2>((w & k.mlo) | k.magic), one, zl), pair(bitcast<h2>((w & k.mhi) | k.magic), sixteenth, zh),
                pair(bitcast<h2>((w8 & k.mlo) | k.magic), one, zl), pair(bitcast<h2>((w8 & k.mhi) | k.magic), sixteenth, zh)};
  }
};

// 16 MT rows x 64 NT columns; KS = 2 K ranges with NW wavefronts that compute and two that copy, and a ring of LDS stages,
// each.  GPB: quantisation groups per K block (1 for group sizes that are multiples of 128, 2 / 4 for 64 / 32).  GLU: half of the
// columns are gate and half the up columns that go with them, with the scales and zero-points of both slabs in a stage.
// LONE: the ring of a workgroup that has its CU for itself.
template <int MT_, int NT_, int GPB_, int ZK, bool GLU_ = false, bool LONE_ = false>
struct RowsCfg {
  static constexpr bool GLU = GLU_;
  static_assert(!GLU || (NT_ == 2 && GPB_ == 1), "64 and 64 columns, one group");
  static constexpr int MT = MT_, NW = 4, NT = NT_, KS = 2, GPB = GPB_;
  static constexpr int BM = 16 * MT, BN = 16 * NW * NT, CW = NW * KS, THREADS = 64 * (CW + 2 * KS);
  static constexpr int A_BYTES = BM * 256, W_BYTES = 1024 * NW * NT, HV = GLU ? 2 : 1,
                       S_BYTES = 256 * GPB * HV, Z_BYTES = (ZK == MI355Q_ZP_PRESCALED ? 256 : 64) * GPB * HV;
  static constexpr int W_OFF = A_BYTES, S_OFF = W_OFF + W_BYTES, Z_OFF = S_OFF + S_BYTES, STAGE = Z_OFF + Z_BYTES;
  static constexpr int XC = A_BYTES / 2048, WC = NW * NT / 2, NC = XC + WC + 1;   // copies of a copying wavefront per stage
  // two workgroups per CU where two stages fit so.  (With two workgroups deeper rings did not gain: the copies are bound by their rate.  One alone has a stage
  // of each range on its way then, and gains by another, but not by a third)
  static constexpr int MOST = LONE_ ? 3 : 4;
  static constexpr int PAIR = !LONE_ && 2 * KS * STAGE <= 80 * 1024 ? 1 : 0, ROOM = (PAIR ? 80 : 159) * 1024 / (KS * STAGE);
  static constexpr int D = ROOM < MOST ? ROOM : MOST, RING = D * STAGE;
  static_assert(XC * 2048 == A_BYTES && WC * 2 == NW * NT && WC <= 4 && D >= 2, "whole copies, a ring");
  static_assert((D - 1) * NC < 64, "copies in flight that the wait can count");
};

// The tile of rows m0 .. and column tile tn over K blocks g0 .. g0 + ng - 1.  GROUPED: rows are the slots ids[0 ..] of one
// expert, gathered from row id / topk of x and stored to row id of the output, times the slot's routing weight.
template <int DT, int ZK, typename C, bool GROUPED>
__device__ __forceinline__ void rows_tile(const RowsArgs& a, const int32_t* ids, int m0, int tn, int g0, int ng) {
  typedef RowsMma<DT> MM;
  constexpr int MT = C::MT, NW = C::NW, NT = C::NT, KS = C::KS, GPB = C::GPB, D = C::D, STAGE = C::STAGE;
  // A operands one K step ahead where the registers are there (else the compiler places the reads, and spills nothing)
  constexpr bool AHEAD = DT == MI355Q_F16 ? MT * NT <= 8 : MT * NT <= (C::PAIR ? 3 : 8);
  extern __shared__ __align__(16) unsigned char lds[];
  const int tid = threadIdx.x, lane = tid & 63, wg = __builtin_amdgcn_readfirstlane(tid >> 6);
  const bool copies = wg >= C::CW;
  const int wave = copies ? (wg - C::CW) % 2 : wg % NW, ks = copies ? (wg - C::CW) / 2 : wg / NW;
  const int c = lane & 15, kq = lane >> 4;
  const int M = a.M, N = a.N, K = a.K, G = K >> 7;
  constexpr bool GLU = C::GLU;
  // 128-column slab (GLU: of the gate columns; the up columns' is N / 256 further), first of the workgroup's 16-column tiles in it
  const int slab = GLU ? tn >> 1 : tn * NW * NT >> 3, t0 = GLU ? 4 * (tn & 1) : tn * NW * NT & 7;
  const int nk = (ng + KS - 1) / KS;                  // ... of each of its ranges (the last may hold fewer, even none)
  const int mine = min(ng - ks * nk, nk);

  f4 acc[MT][NT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[mt][t] = (f4){0.f, 0.f, 0.f, 0.f};

  if (copies) {
    // x: 4 rows of 256 bytes per copy; lane = 16 * row + position, position p of row r receives chunk p ^ (r & 15)
    uint32_t xo[C::XC];
#pragma unroll
    for (int p = 0; p < C::XC; ++p) {
      const int r = 4 * (wave + 2 * p) + (lane >> 4);
      const int row = GROUPED ? min(ids[r], a.numel - 1) / a.topk : min(m0 + r, M - 1);   // (pads read a valid row)
      xo[p] = ((uint32_t)row * (uint32_t)K + 8u * (uint32_t)((lane & 15) ^ (r & 15))) * 2u;
    }
    const uint32_t lane16 = (uint32_t)lane * 16u;
    int kb = min(g0 + ks * nk, G - 1);                // the K block that the next copies are of
    const int klast = max(g0 + ks * nk + mine - 1, kb);
    const char* xg = (const char*)a.x + (size_t)kb * 256;
    const char* qg = (const char*)a.qw + ((size_t)(slab + (GLU ? wave * (N >> 8) : 0)) * G + kb) * 8192 + (t0 + (GLU ? 0 : wave * C::WC)) * 1024;
    // the first wavefront of the range copies the scales, the second the zero-points (without any, the scales again: both
    // have the same number of copies to wait for)
    const bool packed = ZK == MI355Q_ZP_PACKED && wave == 1, zwave = ZK != MI355Q_ZP_NONE && wave == 1;
    const uint32_t szrow = packed ? (uint32_t)N / 2 : (uint32_t)N * 2;
    const uint32_t sznext = GLU ? szrow / 2 : szrow;     // from one group's row to the next one's, or from gate to up
    const uint32_t szoff = packed ? (uint32_t)(lane & 3) * 16u + (uint32_t)(lane >> 2) * sznext
                                  : (uint32_t)(lane & 15) * 16u + (uint32_t)(lane >> 4) * sznext;
    const int szlanes = (packed ? 4 : 16) * GPB * C::HV;
    const char* const szg = zwave ? a.zeros + (packed ? 64 : 256) * slab : (const char*)a.scales + 256 * slab;
    const uint32_t szlds = zwave ? C::Z_OFF : C::S_OFF;
    const uint32_t ring = __builtin_amdgcn_readfirstlane((uint32_t)(size_t)(__attribute__((address_space(3))) unsigned char*)lds) + ks * C::RING;
    auto copy_stage = [&](int slot) {
      const uint32_t sb = ring + (uint32_t)(slot * STAGE);
#pragma unroll
      for (int p = 0; p < C::XC; ++p) lds_copy16(xo[p], xg, sb, (uint32_t)((wave + 2 * p) * 1024));
      lds_copy16(lane16, qg, sb, (uint32_t)(C::W_OFF + wave * C::WC * 1024));
      if constexpr (C::WC > 1) lds_copy16_next<1024>(lane16, qg);
      if constexpr (C::WC > 2) lds_copy16_next<2048>(lane16, qg);
      if constexpr (C::WC > 3) lds_copy16_next<3072>(lane16, qg);
      const uint32_t row = GPB > 1 ? (uint32_t)kb * GPB : a.gpk_magic ? (uint32_t)(((uint64_t)kb * a.gpk_magic) >> 32) : (uint32_t)kb;
      if (lane < szlanes) lds_copy16(szoff, szg + (size_t)row * szrow, sb, szlds);
      if (kb < klast) {                               // (past the end: a re-read into a stage nobody reads)
        ++kb;
        xg += 256;
        qg += 8192;
      }
    };
#pragma unroll
    for (int d = 0; d < D - 1; ++d) copy_stage(d);
    int slot = 0;
    for (int i = 0; i < nk; ++i) {
      asm volatile("s_waitcnt vmcnt(%0)" : : "n"((D - 2) * C::NC) : "memory");   // the copies of K block i have landed
      __builtin_amdgcn_s_barrier();                   // ... everybody's, and nobody reads K block i - 1 any more
      copy_stage(slot == 0 ? D - 1 : slot - 1);
      slot = slot + 1 == D ? 0 : slot + 1;
    }
    asm volatile("s_waitcnt vmcnt(0)" : : : "memory");   // no copy may still be writing LDS
  } else {
    uint32_t a_pos[4];
#pragma unroll
    for (int st = 0; st < 4; ++st) a_pos[st] = (uint32_t)(c * 256 + ((4 * st + kq) ^ c) * 16);
    RowsDq dq = {0x64006400u, 0x000f000fu, 0x00f000f0u};
    asm volatile("" : "+v"(dq.magic));
    asm volatile("" : "+s"(dq.mlo));
    asm volatile("" : "+s"(dq.mhi));
    int slot = 0;
    for (int i = 0; i < nk; ++i) {
      asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");   // no LDS read of the stage before is open
      __builtin_amdgcn_s_barrier();
      asm volatile("" : : : "memory");
      if (i < mine) {
        const unsigned char* st = lds + ks * C::RING + slot * STAGE;
        u4 w[NT], av[2][MT];
        float sc[NT][GPB];
        _Float16 zlo[NT][GPB], zhi[NT][GPB];
        uint32_t rests = 0;                             // not 0: a pre-scaled zero-point is no integer times the scale
        uint32_t zw[GPB];
#pragma unroll
        for (int t = 0; t < NT; ++t) w[t] = *(const u4*)(st + C::W_OFF + (wave * NT + t) * 1024 + lane * 16);
#pragma unroll
        for (int g = 0; g < GPB; ++g)
          zw[g] = ZK == MI355Q_ZP_PACKED ? *(const uint32_t*)(st + C::Z_OFF + 64 * (GLU ? wave >> 1 : g) + c * 4) : 0x88888888u;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) av[0][mt] = *(const u4*)(st + a_pos[0] + mt * 4096);
#pragma unroll
        for (int t = 0; t < NT; ++t) {
          const int tile = t0 + (GLU ? wave & 1 : wave) * NT + t;
#pragma unroll
          for (int g = 0; g < GPB; ++g) {
            sc[t][g] = Elem<DT>::to_f32(*(const uint16_t*)(st + C::S_OFF + 256 * (GLU ? wave >> 1 : g) + (8 * c + tile) * 2));
            if constexpr (ZK == MI355Q_ZP_PRESCALED) {
              const uint16_t zs = *(const uint16_t*)(st + C::Z_OFF + 256 * g + (8 * c + tile) * 2);
              const float zf = prescaled_zero<DT>(zs, sc[t][g]);
              zlo[t][g] = (_Float16)(1024.0f + zf);
              zhi[t][g] = (_Float16)(64.0f + zf);
              rests |= prescaled_differs<DT>(zs, zf, sc[t][g]);
            } else {                                     // fp16 bit patterns directly
              const uint32_t z = (zw[g] >> (4 * tile)) & 15u;
              zlo[t][g] = bitcast<_Float16>((uint16_t)(0x6400u | z));
              zhi[t][g] = bitcast<_Float16>((uint16_t)(0x5400u | (z << 4)));
            }
          }
        }
        f4 part[MT][NT];
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          const int g = s * GPB / 4;
          if (!AHEAD && s > 0) {
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) av[s & 1][mt] = *(const u4*)(st + a_pos[s] + mt * 4096);
          }
          if (AHEAD && s < 3) {
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) av[(s + 1) & 1][mt] = *(const u4*)(st + a_pos[s + 1] + mt * 4096);
          }
          u4 b[NT];
#pragma unroll
          for (int t = 0; t < NT; ++t) b[t] = MM::dequant(w[t][s], zlo[t][g], zhi[t][g], dq);
          if constexpr (AHEAD) asm volatile("" : : : "memory");   // (keeps the reads of the next K step above this one's matrix instructions)
#pragma unroll
          for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int t = 0; t < NT; ++t)
              part[mt][t] = MM::run(av[s & 1][mt], b[t], s % (4 / GPB) == 0 ? (f4){0.f, 0.f, 0.f, 0.f} : part[mt][t]);
          if ((s + 1) % (4 / GPB) == 0) {
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
#pragma unroll
              for (int t = 0; t < NT; ++t) acc[mt][t] += sc[t][g] * part[mt][t];
          }
        }
        if constexpr (ZK == MI355Q_ZP_PRESCALED) {
          // (rare: a checkpoint whose zero-points are no integers) what they hold beyond them times the sum of the group's
          // activations, one matrix instruction with a B operand of ones per K step.  Everything is read from LDS again, so
          // that the loop above has its registers for itself.
          if (__any(rests != 0)) {
            asm volatile("" : : : "memory");
            const uint32_t one = DT == MI355Q_F16 ? 0x3c003c00u : 0x3f803f80u;
            const u4 ones = {one, one, one, one};
#pragma unroll
            for (int g = 0; g < GPB; ++g) {
              float rest[NT];
#pragma unroll
              for (int t = 0; t < NT; ++t) {
                const unsigned char* const q = st + 256 * g + (8 * c + t0 + wave * NT + t) * 2;
                rest[t] = prescaled_rest<DT>(*(const uint16_t*)(q + C::Z_OFF), Elem<DT>::to_f32(*(const uint16_t*)(q + C::S_OFF)));
              }
#pragma unroll
              for (int mt = 0; mt < MT; ++mt) {
                f4 xs = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int s = g * (4 / GPB); s < (g + 1) * (4 / GPB); ++s) xs = MM::run(*(const u4*)(st + a_pos[s] + mt * 4096), ones, xs);
#pragma unroll
                for (int t = 0; t < NT; ++t)
                  if (rest[t] != 0.0f) acc[mt][t] -= rest[t] * xs;
                asm volatile("" : : : "memory");
              }
            }
          }
        }
      }
      slot = slot + 1 == D ? 0 : slot + 1;
    }
    asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");
  }
  __builtin_amdgcn_s_barrier();
  asm volatile("" : : : "memory");

  // through LDS: a lane holds one column of 4 rows per row tile (columns 8 apart in memory), a wavefront's store should
  // hold neighbours.  Tile column j = TC * c + tile is column 8 * (j / TC) + t0 + j % TC of the slab.
  constexpr int EP = C::BN * 4 + 16, TC = NW * NT, Q = TC / 4;         // bytes per tile row; quads of columns per c
  static_assert(C::BM * EP <= C::RING, "the output tile fits in the ring");
  if (!copies) {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          *(float*)(lds + ks * C::RING + (mt * 16 + 4 * kq + i) * EP + (TC * c + wave * NT + t) * 4) = acc[mt][t][i];
  }
  __syncthreads();
  if constexpr (GLU) {
    // tile columns 8 c .. are four gate and the four up columns that go with them
    const int gc = tid % 16;
    for (int r = tid / 16; r < C::BM; r += C::THREADS / 16) {
      const int m = ids[r];
      if (m >= a.numel) continue;
      uint2 o[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        f4 v = *(const f4*)(lds + r * EP + (2 * gc + h) * 16);
#pragma unroll
        for (int k = 1; k < KS; ++k) v += *(const f4*)(lds + k * C::RING + r * EP + (2 * gc + h) * 16);
        o[h].x = (uint32_t)Elem<DT>::from_f32(v[0] + 0.f) | ((uint32_t)Elem<DT>::from_f32(v[1] + 0.f) << 16);
        o[h].y = (uint32_t)Elem<DT>::from_f32(v[2] + 0.f) | ((uint32_t)Elem<DT>::from_f32(v[3] + 0.f) << 16);
      }
      *(uint2*)(a.out + (size_t)m * (N >> 1) + 128 * slab + 8 * gc + t0) = make_uint2(silu_mul16x2<DT>(o[0].x, o[1].x), silu_mul16x2<DT>(o[0].y, o[1].y));
    }
    return;
  }
  constexpr int TPR = C::BN / 4;                      // threads per row
  const int q = tid % TPR, n = 128 * slab + 8 * (q / Q) + t0 + 4 * (q % Q);
  float bs[4] = {0.f, 0.f, 0.f, 0.f};
  if (!GROUPED && a.bias && !a.partial) {
    const uint2 bw = *(const uint2*)(a.bias + n);
    bs[0] = Elem<DT>::to_f32((uint16_t)(bw.x & 0xffffu)); bs[1] = Elem<DT>::to_f32((uint16_t)(bw.x >> 16));
    bs[2] = Elem<DT>::to_f32((uint16_t)(bw.y & 0xffffu)); bs[3] = Elem<DT>::to_f32((uint16_t)(bw.y >> 16));
  }
  for (int r = tid / TPR; r < C::BM; r += C::THREADS / TPR) {
    const int m = GROUPED ? ids[r] : m0 + r;
    if (m >= (GROUPED ? a.numel : M)) {
      if (GROUPED) continue;
      break;
    }
    f4 v = *(const f4*)(lds + r * EP + q * 16);
#pragma unroll
    for (int k = 1; k < KS; ++k) v += *(const f4*)(lds + k * C::RING + r * EP + q * 16);
    if (!GROUPED && a.partial) {
      *(f4*)(a.partial + ((size_t)blockIdx.y * M + m) * N + n) = v;
    } else {
      if (GROUPED && a.topk_weights) v *= a.topk_weights[m];
      uint2 o;
      o.x = (uint32_t)Elem<DT>::from_f32(v[0] + bs[0]) | ((uint32_t)Elem<DT>::from_f32(v[1] + bs[1]) << 16);
      o.y = (uint32_t)Elem<DT>::from_f32(v[2] + bs[2]) | ((uint32_t)Elem<DT>::from_f32(v[3] + bs[3]) << 16);
      *(uint2*)(a.out + (size_t)m * N + n) = o;
    }
  }
}

template <int DT, int ZK, typename C>
__global__ void __launch_bounds__(C::THREADS, (C::PAIR + 1) * C::THREADS / 256)
w4a16_rows_kernel(RowsArgs a) {
  const int t = xcd_tile();
  const int tn = t / a.mtiles, tm = t - tn * a.mtiles;
  const int g0 = (int)blockIdx.y * a.kper;
  rows_tile<DT, ZK, C, false>(a, nullptr, tm * C::BM, tn, g0, min((a.K >> 7) - g0, a.kper));
}

// Blocks of up to 16 MAX slots: a block takes the tile of as many row tiles as hold real slots (they come first).  GLU: the columns are gate
// and up, and what is stored ([numel, N / 2]) is what silu_and_mul makes of the sums that would have been: its pass and half of the stores are
// saved (us for a whole layer, 86 .. 224 of which 4 .. 7 were that pass: 79.0 -> 74.9, 111.6 -> 107.3, 171.7 -> 168.4).
template <int DT, int ZK, int GPB, int MAX, bool GLU>
__global__ void __launch_bounds__(768, (RowsCfg<MAX, 2, GPB, ZK, GLU>::PAIR + 1) * 3)
w4a16_rows_grouped_kernel(RowsArgs a) {
  const int base = blockIdx.y * a.block;
  if (base >= *a.npp) return;                         // block beyond the padded ids
  const int32_t* const ids = a.sorted_ids + base;
  const int lane = threadIdx.x & 63, tn = blockIdx.x;
  const unsigned long long real = __ballot(lane < a.block && ids[min(lane, a.block - 1)] < a.numel);
  if (!real) return;                                  // pads only
  const long e = a.expert_ids[blockIdx.y];
  if (e < 0 || e >= a.E) {                            // not one of this rank's experts: zero rows, no weights read
    if (GLU) zero_block_columns(a.out, ids, a.block, a.numel, a.N >> 1, tn * 64, 64, 768);
    else zero_block_columns(a.out, ids, a.block, a.numel, a.N, tn * 128, 128, 768);
    return;
  }
  a.qw = (const u4*)((const char*)a.qw + e * a.w_stride);
  a.scales = (const uint16_t*)((const char*)a.scales + e * a.s_stride);
  if (a.zeros) a.zeros += e * a.z_stride;
  const int tiles = __builtin_amdgcn_readfirstlane((64 - __builtin_clzll(real) + 15) >> 4), G = a.K >> 7;
  if (tiles == 1) return rows_tile<DT, ZK, RowsCfg<1, 2, GPB, ZK, GLU>, true>(a, ids, 0, tn, 0, G);
  if (MAX == 2 || tiles == 2) return rows_tile<DT, ZK, RowsCfg<2, 2, GPB, ZK, GLU>, true>(a, ids, 0, tn, 0, G);
  if constexpr (MAX > 2) {
    if (tiles == 3) return rows_tile<DT, ZK, RowsCfg<3, 2, GPB, ZK, GLU>, true>(a, ids, 0, tn, 0, G);
    rows_tile<DT, ZK, RowsCfg<4, 2, GPB, ZK, GLU>, true>(a, ids, 0, tn, 0, G);
  }
}

template <int DT, int ZK, typename C>
int launch_rows(RowsArgs a, int splits, const void* bias, int dtype, hipStream_t st) {
  const int G = a.K / 128;
  a.mtiles = (a.M + C::BM - 1) / C::BM;
  a.kper = (G + splits - 1) / splits;
  splits = (G + a.kper - 1) / a.kper;                 // no empty ranges
  if (splits <= 1) a.partial = nullptr;
  const size_t shmem = (size_t)C::KS * C::RING;
  static hipError_t attr = hipFuncSetAttribute((const void*)w4a16_rows_kernel<DT, ZK, C>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)shmem);
  MQ_REQUIRE(attr == hipSuccess, "w4a16_gemm(rows): cannot reserve %zu bytes of LDS: %s", shmem, hipGetErrorString(attr));
  hipLaunchKernelGGL((w4a16_rows_kernel<DT, ZK, C>), dim3((unsigned)(a.mtiles * (a.N / C::BN)), (unsigned)splits), dim3(C::THREADS), shmem, st, a);
  MQ_LAUNCH_CHECK("w4a16_gemm(rows)");
  if (splits > 1) return w4a16_splitk_reduce_launch(a.out, a.partial, bias, a.M, a.N, splits, dtype, st);
  return 0;
}

template <int DT, int ZK, int GPB>
int launch_rows_cfg(const RowsArgs& a, int mt, int nt, int splits, const void* bias, int dtype, hipStream_t st) {
  // no more workgroups than CUs: LONE, but for 32 x 128 with bf16, whose arithmetic fills the wait (us, there / here: 4096 x 28672 at 20 rows 17.5 / 18.7, 14336 x 8192 at 18
  // 21.4 / 22.0, 3584 x 18944 at 24 16.6 / 17.0; only 8192 x 28672 and 5120 x 27648 below 21 rows gain, 37.9 / 34.7)
  const bool lone = (long)((a.M + 16 * mt - 1) / (16 * mt)) * (a.N / (64 * nt)) * splits <= device_cu_count();
#define MQ_CFG(MT, NT)                                                                                                                  \
  if (mt == MT && nt == NT) {                                                                                                           \
    if constexpr (RowsCfg<MT, NT, GPB, ZK>::PAIR && (NT == 1 || DT == MI355Q_F16))                                                      \
      if (lone) return launch_rows<DT, ZK, RowsCfg<MT, NT, GPB, ZK, false, true>>(a, splits, bias, dtype, st);                          \
    return launch_rows<DT, ZK, RowsCfg<MT, NT, GPB, ZK>>(a, splits, bias, dtype, st);                                                   \
  }
  MQ_CFG(2, 1) MQ_CFG(3, 1) MQ_CFG(4, 1)
  MQ_CFG(2, 2) MQ_CFG(3, 2) MQ_CFG(4, 2) MQ_CFG(5, 2) MQ_CFG(6, 2)
#undef MQ_CFG
  MQ_REQUIRE(false, "w4a16_gemm(rows): no tile of %d x %d", 16 * mt, 64 * nt);
}

// ---- the choice of tile and K split: the cheapest by a price model in microseconds.  Per tile: a K block of each of its two
// ranges, for a workgroup with its CU for itself (`lone`, where that is another ring than that of two), else for the first one on its CU and added for a
// second one beside it (tiles of 64 columns and 32 x 128 fit two).  Above 128 rows, where the other kernels' prices are compared with this one: fitted to 3400
// measurements (15 layer shapes, 20..2048 rows, 1..12 ranges, weights cold in the caches; rms error 5 %), without rings of their own for lone workgroups.  Up to
// 128 rows: to the launches of 42 layers with each type (18 .. 128 rows, up to eight ranges, weights from memory; rms errors 6 and 5 %), and with fp16 then moved until the
// tiles taken over 34 layers were right with weights from memory and from the Infinity Cache both, K ranges charged 0.2 us for their second launch (3584 x 37888
// at 33 rows, by the first fit and now: 31.3 / 32.1 us from memory, 33.2 / 27.9 from the cache).  The tile taken loses 0.2 / 0.2 % (fp16 / bf16) to the best one on average,
// 7 % at worst, and against the prices above 128 rows gains 3.6 / 3.1 % from memory and 1.6 / 1.3 % from the cache.
struct RowsPrice {
  int mt, nt;
  double one, more, lone;
};
struct RowsModel {
  RowsPrice tiles[8];
  double base, round, split, split_mn;
  double alone;               // share of a step that goes away as the chip empties (the caches and memory are shared)
  double second;              // share of the second workgroup's price that grows with how many CUs hold two
  double stream;              // bytes of weights per microsecond
};
constexpr RowsModel kRows[3] = {
    {{{2, 1, 0.422, 0.388, 0.422}, {3, 1, 0.600, 0.500, 0.600}, {4, 1, 0.700, 0, 0}, {2, 2, 0.773, 0.594, 0.773},
      {3, 2, 0.956, 0, 0}, {4, 2, 1.173, 0, 0}, {5, 2, 1.333, 0, 0}, {6, 2, 1.555, 0, 0}},
     3.57, 1.10, 2.18, 1.56, 0.283, 0.388, 4.23e6},
    {{{2, 1, 0.332, 0.643, 0.458}, {3, 1, 0.705, 0.364, 0.589}, {4, 1, 0.736, 0, 0}, {2, 2, 0.650, 0.672, 0.872},
      {3, 2, 0.959, 0, 0}, {4, 2, 1.135, 0, 0}, {5, 2, 1.232, 0, 0}, {6, 2, 1.545, 0, 0}},
     3.37, 1.25, 1.66, 2.97, 0.175, 0.249, 4.39e6},
    {{{2, 1, 0.464, 0.522, 0.511}, {3, 1, 0.605, 0.541, 0.640}, {4, 1, 0.750, 0, 0}, {2, 2, 0.597, 1.143, 0.908},
      {3, 2, 1.137, 0, 0}, {4, 2, 1.258, 0, 0}, {5, 2, 1.519, 0, 0}, {6, 2, 1.599, 0, 0}},
     4.05, 1.45, 1.79, 1.95, 0.155, 0.149, 4.04e6}};
const RowsModel& rows_model(int M, bool bf16) { return kRows[M > 128 ? 0 : bf16 ? 2 : 1]; }

struct RowsPlan {
  int mt, nt, splits;
  size_t bytes;                             // partial sums
  double price;
};

RowsPlan rows_make_plan(const RowsModel& m, int M, int K, int N, bool split) {
  RowsPlan best = {0, 0, 1, 0, 1e30};
  const int KB = K / 128;
  const long cus = device_cu_count();
  const double stream = std::pow((double)K * N / 2 / m.stream, 4);
  for (const RowsPrice& p : m.tiles) {
    const int bm = 16 * p.mt, bn = 64 * p.nt;
    if (p.mt > 2 && M <= bm - 16) continue;
    const long tiles = (long)((M + bm - 1) / bm) * (N / bn), res = p.more > 0 ? 2 : 1;
    for (int s = 1; s <= (split ? 12 : 1); ++s) {
      const int kper = (KB + s - 1) / s;
      if (s > 1 && ((KB + kper - 1) / kper != s || kper < 8)) continue;
      const size_t bytes = s > 1 ? (size_t)s * M * N * 4 : 0;
      if (bytes > ((size_t)31 << 20)) continue;       // (fits the fixed scratch of callers that cannot allocate, too)
      const long full = tiles * s / (res * cus), rest = tiles * s % (res * cus);
      const double one = p.lone > 0 && tiles * s <= cus ? p.lone : p.one;
      double steps = full * (p.one + p.more * (res - 1));
      if (rest) steps += one * (1 - m.alone * (1 - (double)std::min(rest, cus) / cus));
      if (rest > cus) steps += p.more * ((double)(rest - cus) / cus * m.second + 1 - m.second);
      double t = std::sqrt(std::sqrt(std::pow(steps * ((kper + 1) / 2), 4) + stream)) + m.base + m.round * (full + (rest > 0) - 1);
      if (s > 1) t += m.split + m.split_mn * 1e-6 * s * M * N;
      if (t < best.price) best = {p.mt, p.nt, s, bytes, t};
    }
  }
  return best;
}

// of fp16 and of bf16 (together: whoever sizes a workspace asks for both)
struct RowsPlans {
  RowsPlan of[2];
};
RowsPlans rows_plans(int M, int K, int N) {
  return cached_plan(0, M, N, K, [](int, int M, int N, int K) {
    const RowsPlan f16 = rows_make_plan(rows_model(M, false), M, K, N, true);
    return RowsPlans{{f16, M > 128 ? f16 : rows_make_plan(rows_model(M, true), M, K, N, true)}};
  });
}

template <int DT, int ZK, int GPB, int MAX, bool GLU = false>
int launch_rows_grouped(const RowsArgs& a, int max_blocks, hipStream_t st) {
  size_t shmem = 0;
  for (size_t b : {(size_t)RowsCfg<1, 2, GPB, ZK, GLU>::RING, (size_t)RowsCfg<2, 2, GPB, ZK, GLU>::RING, MAX > 2 ? (size_t)RowsCfg<3, 2, GPB, ZK, GLU>::RING : 0,
                   MAX > 2 ? (size_t)RowsCfg<4, 2, GPB, ZK, GLU>::RING : 0})
    shmem = std::max(shmem, 2 * b);
  static hipError_t attr = hipFuncSetAttribute((const void*)w4a16_rows_grouped_kernel<DT, ZK, GPB, MAX, GLU>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)shmem);
  MQ_REQUIRE(attr == hipSuccess, "moe_w4a16(rows): cannot reserve %zu bytes of LDS: %s", shmem, hipGetErrorString(attr));
  hipLaunchKernelGGL((w4a16_rows_grouped_kernel<DT, ZK, GPB, MAX, GLU>), dim3((unsigned)(a.N / 128), (unsigned)max_blocks), dim3(768), shmem, st, a);
  MQ_LAUNCH_CHECK("moe_w4a16(rows)");
  return 0;
}

}  // namespace

double w4a16_rows_price(int M, int K, int N) { return rows_plans(M, K, N).of[0].price; }
double w4a16_wide_price(int M, int K, int N, int group_size, int zeros_kind, bool bf16);     // us of the 64-row tiles and the ring kernels

// Whether this kernel is the one to take.
//  - Up to 16 rows: the streaming kernel, except for groups of 64 and 32 on small layers, where four scale rows per K block
//    keep it from its rate (4096 x 4096, groups of 64, 1 / 16 rows: 9.1 / 10.2 -> 7.8 / 8.3 us, 2048 x 2048 8.3 / 8.7 -> 6.5 / 6.7;
//    4096 x 28672, bf16: 16.2 against 19.8).
//  - 17..32 rows: there the streaming kernel takes two row tiles and stays ahead on groups of 128 while the layer is small in both directions (us at 24 rows, fp16,
//    there / here: 4096 x 6144 8.8 / 9.3, 2048 x 7168 6.0 / 6.5, 4096 x 4096 8.3 / 8.2; from 8192 columns 1408 x 19328 10.3 / 8.2, 4096 x 12288 11.8 / 11.0, 2560 x 8960
//    8.3 / 7.7; from K 5120 5248 x 3840 8.9 / 8.7), and with bf16, whose operands cost more here, up to 16384 columns (4096 x 12288 11.9 / 12.5; 2432 x 18944
//    14.6 / 13.5).  K ranges here are a second launch, which the streaming kernel does without: 3 us more of host time in a call (3.3 -> 6.1, 7168 x 2560 at 30), so they have to
//    be worth that.  14336 x 4096 14.7 / 13.3 and 6144 x 2048 8.6 / 7.6 are not (a whole layer of 2560 x 14336 and 7168 x 2560 at 30, launched call by call, 39.4 -> 41.7);
//    the largest layers are (from 67 million weights with fp16, 100 million with bf16).
//  - Pre-scaled zero-points up to 64 rows: the streaming kernel, which uses z * s as it is.
//  - To 128 rows: always.  Above: where its price is below that of the kernels with larger tiles, which read and dequantise the
//    weights fewer times, as those operands run there.
bool w4a16_rows_wanted(int M, int K, int N, int group_size, int zeros_kind, int dtype) {
  const bool small = group_size % 128 != 0;
  const long w = (long)K * N;
  if (small && group_size != 64 && group_size != 32) return false;
  if (M > 4096 || (size_t)M * K * 2 >= ((size_t)1 << 32)) return false;
  if (zeros_kind == MI355Q_ZP_PRESCALED && M <= 64) return false;
  if (M <= 16) return small && w <= (1L << 25);
  if (M <= 32) {
    const bool bf = dtype == MI355Q_BF16;
    if (small || w >= (bf ? 3L << 25 : 1L << 26)) return true;
    return (bf ? N >= 16384 : N >= 8192 || K >= 5120) && rows_plans(M, K, N).of[bf].splits == 1;
  }
  if (M <= 128) return true;
  // (the price, corrected for the size of the output and the rows by 255 launches with fp16 rows and 177 with bf16, rms errors 4.6 and 3 %.  The
  // pick loses 0.1 / 0.2 % (fp16 / bf16) to the best of the three kernels over 23 layers at 144 .. 2048 rows, 15 % at worst, where prices
  // tie: fp16 5120 x 13824 at 200 rows 53.7 us on the tiles, 46.1 here; 3584 x 37888 at 144 59.5 / 64.  The
  // loops that are not pipelined by 1300 launches, 0.2 %: bf16 with groups of 64 4096 x 6144 at 1536 100 us here, 142 there, with groups of 32
  // 117 / 180, bf16 rows that are not staged 28672 x 8192 at 170 102 / 124, fp16 with groups of 32 3584 x 37888 at 256 119 / 159.)
  const bool bf16 = dtype == MI355Q_BF16;
  const double corrected = w4a16_rows_price(M, K, N) * (bf16 ? 1.023 + 14e-6 * M : 0.881 + 66e-6 * M) + 0.78e-6 * M * N;
  return corrected < w4a16_wide_price(M, K, N, group_size, zeros_kind, bf16);
}

// (of either type)
size_t w4a16_rows_workspace_bytes(int M, int K, int N) {
  if (M > 4096) return 0;
  const RowsPlans p = rows_plans(M, K, N);
  return std::max(p.of[0].bytes, p.of[1].bytes);
}

// mt 0: the plan, unsplit where the workspace does not hold the partial sums; else 16 mt rows x 64 nt columns, K in `splits` ranges
int w4a16_rows_launch(void* out, const void* x, const int32_t* qweight, const void* scales, const void* zeros, int zeros_kind,
                      const void* bias, int M, int K, int N, int group_size, int dtype, void* workspace, size_t workspace_bytes,
                      int mt, int nt, int splits, hipStream_t st) {
  if (!mt) {
    const bool bf16 = dtype == MI355Q_BF16;
    RowsPlan p = rows_plans(M, K, N).of[bf16];
    if (p.bytes > (workspace ? workspace_bytes : 0)) p = rows_make_plan(rows_model(M, bf16), M, K, N, false);
    mt = p.mt;
    nt = p.nt;
    splits = p.splits;
  }
  splits = std::max(1, std::min(splits, K / 128));
  if (splits > 1 && (!workspace || workspace_bytes < (size_t)splits * M * N * 4)) splits = 1;
  MQ_REQUIRE((size_t)M * K * 2 < ((size_t)1 << 32), "w4a16_gemm: activation matrix %d x %d is 4 GiB or more", M, K);
  MQ_REQUIRE(group_size % 128 == 0 || group_size == 64 || group_size == 32, "w4a16_gemm(rows): group size %d", group_size);
  RowsArgs a = {};
  a.out = (uint16_t*)out; a.x = (const uint16_t*)x; a.qw = (const u4*)qweight; a.scales = (const uint16_t*)scales;
  a.zeros = (const char*)zeros; a.bias = (const uint16_t*)bias;
  a.M = M; a.K = K; a.N = N;
  const uint32_t gpk = group_size >= 128 ? (uint32_t)group_size / 128u : 1u;
  a.gpk_magic = gpk > 1 ? (uint32_t)((((uint64_t)1 << 32) + gpk - 1) / gpk) : 0u;
  a.partial = (float*)workspace;
#define MQ_GPB(DT, ZK, GPB) return launch_rows_cfg<DT, ZK, GPB>(a, mt, nt, splits, bias, dtype, st)
#define MQ_ZK(DT, ZK)                       \
  do {                                      \
    if (group_size == 64) MQ_GPB(DT, ZK, 2); \
    if (group_size == 32) MQ_GPB(DT, ZK, 4); \
    MQ_GPB(DT, ZK, 1);                      \
  } while (0)
#define MQ_DT(DT)                                                          \
  do {                                                                     \
    if (zeros_kind == MI355Q_ZP_PACKED) MQ_ZK(DT, MI355Q_ZP_PACKED);       \
    if (zeros_kind == MI355Q_ZP_PRESCALED) MQ_ZK(DT, MI355Q_ZP_PRESCALED); \
    MQ_ZK(DT, MI355Q_ZP_NONE);                                             \
  } while (0)
  if (dtype == MI355Q_F16) MQ_DT(MI355Q_F16);
  MQ_DT(MI355Q_BF16);
#undef MQ_DT
#undef MQ_ZK
#undef MQ_GPB
}

// blocks of 32 or 64 slots of one expert, groups of 64 or multiples of 128
int w4a16_rows_grouped_launch(void* out, const void* x, const int32_t* qweight, const void* scales, const void* zeros, int zeros_kind,
                              const float* topk_weights, const int32_t* sorted_ids, const int32_t* expert_ids, const int32_t* npp,
                              int numel, int topk, int block_size, int max_blocks, int E, int K, int N, int group_size, int dtype,
                              hipStream_t st, bool glu) {
  MQ_REQUIRE(block_size == 32 || block_size == 64, "moe_w4a16(rows): blocks of 32 or 64 slots, got %d", block_size);
  MQ_REQUIRE(group_size % 128 == 0 || group_size == 64, "moe_w4a16(rows): group size %d", group_size);
  RowsArgs a = {};
  a.out = (uint16_t*)out; a.x = (const uint16_t*)x; a.qw = (const u4*)qweight; a.scales = (const uint16_t*)scales;
  a.zeros = (const char*)zeros;
  a.M = numel; a.K = K; a.N = N;
  const uint32_t gpk = group_size >= 128 ? (uint32_t)group_size / 128u : 1u;
  a.gpk_magic = gpk > 1 ? (uint32_t)((((uint64_t)1 << 32) + gpk - 1) / gpk) : 0u;
  a.sorted_ids = sorted_ids; a.expert_ids = expert_ids; a.npp = npp; a.topk_weights = topk_weights;
  a.numel = numel; a.topk = topk; a.E = E; a.block = block_size;
  a.w_stride = (long)K * N / 2;
  a.s_stride = (long)(K / group_size) * N * 2;
  a.z_stride = zeros_kind == MI355Q_ZP_PACKED ? (long)(K / group_size) * N / 2 : a.s_stride;
#define MQ_GLU(DT, ZK)                                                                                                                  \
  return block_size == 32 ? launch_rows_grouped<DT, ZK, 1, 2, true>(a, max_blocks, st) : launch_rows_grouped<DT, ZK, 1, 4, true>(a, max_blocks, st)
  if (glu) {
    MQ_REQUIRE(group_size % 128 == 0 && N % 256 == 0 && zeros_kind != MI355Q_ZP_PRESCALED, "moe_w4a16(rows): gate and up of N=%d, group size %d", N, group_size);
    if (dtype == MI355Q_F16 && zeros_kind == MI355Q_ZP_PACKED) MQ_GLU(MI355Q_F16, MI355Q_ZP_PACKED);
    if (dtype == MI355Q_F16) MQ_GLU(MI355Q_F16, MI355Q_ZP_NONE);
    if (zeros_kind == MI355Q_ZP_PACKED) MQ_GLU(MI355Q_BF16, MI355Q_ZP_PACKED);
    MQ_GLU(MI355Q_BF16, MI355Q_ZP_NONE);
  }
#undef MQ_GLU
#define MQ_MAX(DT, ZK, GPB)                                                                                               \
  return block_size == 32 ? launch_rows_grouped<DT, ZK, GPB, 2>(a, max_blocks, st) : launch_rows_grouped<DT, ZK, GPB, 4>(a, max_blocks, st)
#define MQ_ZK(DT, ZK)                         \
  do {                                        \
    if (group_size == 64) MQ_MAX(DT, ZK, 2);  \
    MQ_MAX(DT, ZK, 1);                        \
  } while (0)
#define MQ_DT(DT)                                                          \
  do {                                                                     \
    if (zeros_kind == MI355Q_ZP_PACKED) MQ_ZK(DT, MI355Q_ZP_PACKED);       \
    if (zeros_kind == MI355Q_ZP_PRESCALED) MQ_ZK(DT, MI355Q_ZP_PRESCALED); \
    MQ_ZK(DT, MI355Q_ZP_NONE);                                             \
  } while (0)
  if (dtype == MI355Q_F16) MQ_DT(MI355Q_F16);
  MQ_DT(MI355Q_BF16);
#undef MQ_DT
#undef MQ_ZK
#undef MQ_MAX
}

}  // namespace mi355q
