// W4A16 GEMM for up to 16 rows over layers that one round of workgroups covers without cutting K between them.
//
// On such a layer (4096 x 4096: 32 KiB of weights per CU) the stream is over before a loop has found its pace: the
// streaming kernel's wavefronts walk eight K blocks of 128, one block ahead of the arithmetic, alone on their SIMD, at 0.5 us a
// block whatever a block carries.  Here a workgroup has 8 or 16 wavefronts and each of them asks for everything it will ever
// read -- up to four K blocks, on deep K to seven -- before it computes the first, in straight-line code, so that one trip to memory covers the
// launch.  What bounds it: launch, that trip and the last stores (a kernel that only reads the weights of 4096 x 4096 takes 2.6 us); from
// nine rows on also the activations, which every workgroup reads in whole through its L1: a row travels 256 bytes at a time
// (16 lanes; four lanes to a row cost the address unit twice as much) and up to four, eight or sixteen rows are asked for, and
// is turned into operands through LDS.
// fp16 operands are the exact integers q - z; bf16 ones 128 + q, whose 128 + z times the sum of the row is taken off
// the fp32 sum of each group.
//
// Measured (us, graph replays, weights warm in the last-level cache / cold, the streaming kernel -> here, fp16, groups of 128): 4096 x 4096 at
// 1 / 4 / 16 rows 5.0 / 5.6 / 5.6 -> 3.5 / 3.5 / 4.7 warm, 6.1 / 6.1 / 6.3 -> 4.0 / 4.1 / 5.4 cold; 4096 x 6144 at 1 / 16 6.0 / 6.2 -> 4.5 / 5.8 and
// 6.7 / 6.9 -> 5.2 / 6.6; 8192 x 8192 at 1 / 8 9.5 / 9.9 -> 8.0 / 8.7 and 10.9 / 10.7 -> 8.4 / 9.2; 1024 x 1024 at 1 2.8 -> 2.3.
#include "moe_slots.h"

#include <algorithm>
#include <cmath>
#include <type_traits>

namespace mi355q {
namespace {

struct DecodeArgs {
  uint16_t* out;
  const uint16_t* x;
  const u4* qw;
  const uint16_t* scales;
  const void* zeros;            // packed int4 or null
  const uint16_t* bias;
  int M, K, N;
  uint32_t gpk_magic;           // ceil(2^32 / K blocks per group); 0: a group is one K block
  int qrows;                    // K / group size
  // grouped (fused-MoE) launches: blockIdx.z = block of 16 sorted token slots, all of one expert
  const int32_t* sorted_ids;    // slot ids, pads >= numel
  const int32_t* expert_ids;    // [blocks]
  const int32_t* npp;           // device scalar: slots after padding
  const float* topk_weights;    // [numel] or null
  int numel, topk, E;
  int id_step, id_bits;         // launches without an alignment: sorted_ids are the slots' experts, int32 per id, bits of an expert
  long w_stride, s_stride, z_stride;   // bytes per expert
  int kper;                     // K blocks per range (blockIdx.y)
  float* partial;               // f32 sums [range][numel][N], without the routing weights; null: write the output
};

template <int DT> struct DecodeMma;
template <> struct DecodeMma<MI355Q_F16> {
  static __device__ __forceinline__ f4 run(const u4& a, const u4& b, f4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(bitcast<h8>(a), bitcast<h8>(b), c, 0, 0, 0);
  }
};
template <> struct DecodeMma<MI355Q_BF16> {
  static __device__ __forceinline__ f4 run(const u4& a, const u4& b, f4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(bitcast<b8>(a), bitcast<b8>(b), c, 0, 0, 0);
  }
};

template <int N>
__device__ __forceinline__ void load_halves(rsrc_t r, uint32_t off, uint32_t* dst) {
  if constexpr (N == 8) {
    const u4 v = buf_load16(r, off);
    dst[0] = v[0]; dst[1] = v[1]; dst[2] = v[2]; dst[3] = v[3];
  } else if constexpr (N == 4) {
    const u2 v = bitcast<u2>(__builtin_amdgcn_raw_buffer_load_b64(r, (int)off, 0, 0));
    dst[0] = v[0]; dst[1] = v[1];
  } else if constexpr (N == 2) {
    dst[0] = __builtin_amdgcn_raw_buffer_load_b32(r, (int)off, 0, 0);
  } else {
    dst[0] = __builtin_amdgcn_raw_buffer_load_b16(r, (int)off, 0, 0);
  }
}

template <int DT, int N>
__device__ __forceinline__ void store_row(uint16_t* out, const uint16_t* bias, const float* v) {
  uint16_t h[N];
#pragma unroll
  for (int t = 0; t < N; ++t) h[t] = Elem<DT>::from_f32(bias ? v[t] + Elem<DT>::to_f32(bias[t]) : v[t]);
  if constexpr (N == 1) {
    const uint32_t val = h[0];
    asm volatile("global_store_short %0, %1, off sc0 sc1" ::"v"(out), "v"(val) : "memory");
  } else if constexpr (N == 2) {
    const uint32_t val = (uint32_t)h[0] | ((uint32_t)h[1] << 16);
    asm volatile("global_store_dword %0, %1, off sc0 sc1" ::"v"(out), "v"(val) : "memory");
  } else if constexpr (N == 4) {
    const u2 val = {(uint32_t)h[0] | ((uint32_t)h[1] << 16), (uint32_t)h[2] | ((uint32_t)h[3] << 16)};
    asm volatile("global_store_dwordx2 %0, %1, off sc0 sc1" ::"v"(out), "v"(val) : "memory");
  } else {
    const u4 val = {(uint32_t)h[0] | ((uint32_t)h[1] << 16), (uint32_t)h[2] | ((uint32_t)h[3] << 16), (uint32_t)h[4] | ((uint32_t)h[5] << 16),
                    (uint32_t)h[6] | ((uint32_t)h[7] << 16)};
    asm volatile("global_store_dwordx4 %0, %1, off sc0 sc1" ::"v"(out), "v"(val) : "memory");
  }
}

// weights, scales and zero-points of one K block: NT tiles of 16 columns (GLU: of NT / 2 in each of two slabs)
template <int NT, int ZK, bool GLU = false>
struct DecodeBlock {
  static constexpr int HW = NT >= 2 ? NT / 2 : 1;
  u4 w[NT];
  uint32_t s[HW], z[ZK == MI355Q_ZP_PRESCALED ? HW : GLU ? 2 : 1];
};
struct DecodeConst {
  uint32_t magic, mlo, mhi;     // (in registers: as literals an and and an or, not one instruction)
};
template <int DT>
__device__ __forceinline__ DecodeConst decode_const() {
  DecodeConst k = {DT == MI355Q_F16 ? 0x64006400u : 0x43004300u, 0x000f000fu, 0x00f000f0u};
  asm volatile("" : "+v"(k.magic));
  asm volatile("" : "+s"(k.mlo));
  asm volatile("" : "+s"(k.mhi));
  return k;
}

template <int DT, int ZK, int NT, bool GLU = false>
__device__ __forceinline__ void decode_block(f4* acc, const u4* x, const DecodeBlock<NT, ZK, GLU>& b, int t0, const DecodeConst& k) {
  typedef DecodeMma<DT> MM;
  constexpr bool SUMS = DT == MI355Q_BF16 || ZK == MI355Q_ZP_PRESCALED;
  f4 xs = {0.f, 0.f, 0.f, 0.f};
  if constexpr (SUMS) {
    const uint32_t one = DT == MI355Q_F16 ? 0x3c003c00u : 0x3f803f80u;
    const u4 ones = {one, one, one, one};
#pragma unroll
    for (int s = 0; s < 4; ++s) xs = MM::run(x[s], ones, xs);
  }
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const float sc = Elem<DT>::to_f32((uint16_t)((t & 1) ? (b.s[t >> 1] >> 16) : (b.s[t >> 1] & 0xffffu)));
    const uint32_t z = ZK == MI355Q_ZP_PRESCALED ? 0u : (b.z[GLU ? 2 * t / NT : 0] >> (4 * (t0 + (GLU ? t % (NT / 2) : t)))) & 15u;
    f4 part;
    if constexpr (DT == MI355Q_F16) {
      const _Float16 zl = bitcast<_Float16>((uint16_t)(0x6400u | z)), zh = bitcast<_Float16>((uint16_t)(0x5400u | (z << 4)));
      const h2 zlo = {zl, zl}, zhi = {zh, zh}, sixteenth = {(_Float16)0.0625f, (_Float16)0.0625f};
      part = (f4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const uint32_t w = b.w[t][s], w8 = w >> 8;
        const h2 r0 = bitcast<h2>((w & k.mlo) | k.magic) - zlo;                                          // 1024 + q
        const h2 r1 = __builtin_elementwise_fma(bitcast<h2>((w & k.mhi) | k.magic), sixteenth, -zhi);    // 1024 + 16 q
        const h2 r2 = bitcast<h2>((w8 & k.mlo) | k.magic) - zlo;
        const h2 r3 = __builtin_elementwise_fma(bitcast<h2>((w8 & k.mhi) | k.magic), sixteenth, -zhi);
        part = MM::run(x[s], (u4){bitcast<uint32_t>(r0), bitcast<uint32_t>(r1), bitcast<uint32_t>(r2), bitcast<uint32_t>(r3)}, part);
      }
    } else {
      part = -(128.0f + (float)z) * xs;
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const uint32_t w = b.w[t][s];
        part = MM::run(x[s], (u4){(w & k.mlo) | k.magic, ((w >> 4) & k.mlo) | k.magic, ((w >> 8) & k.mlo) | k.magic, ((w >> 12) & k.mlo) | k.magic}, part);
      }
    }
    if constexpr (ZK == MI355Q_ZP_PRESCALED) {
      const uint32_t zw = b.z[(t >> 1) < DecodeBlock<NT, ZK, GLU>::HW ? t >> 1 : 0];
      acc[t] += sc * part - Elem<DT>::to_f32((uint16_t)((t & 1) ? (zw >> 16) : (zw & 0xffffu))) * xs;
    } else {
      acc[t] += sc * part;
    }
  }
}

// NT tiles of 16 columns, W wavefronts of up to B K blocks each, up to 4 XN rows
template <int DT, int ZK, int NT, int W, int B, int XN>
__global__ void __launch_bounds__(64 * W, W / 4)
w4a16_decode_kernel(DecodeArgs a) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = lane & 15, kq = lane >> 4;
  constexpr int TG = 8 / NT;
  const int group = xcd_tile(), slab = group / TG, t0 = (group % TG) * NT;
  const int G = a.K >> 7, N = a.N, K = a.K;
  const int ncol8 = 128 * slab + 8 * c, ncol = ncol8 + t0;
  constexpr int RED = W * 4 * NT * 64 * 4, XL = W * 1024 * XN;    // x: 16 lanes to a row, four rows per load
  __shared__ __align__(16) unsigned char lds[RED > XL ? RED : XL];

  struct Block : DecodeBlock<NT, ZK> {
    u4 x[XN];
  };
  const rsrc_t wres = make_rsrc(a.qw + (size_t)slab * G * 512, (uint32_t)G * 8192u);
  const rsrc_t sres = make_rsrc(a.scales, (uint32_t)a.qrows * N * 2u);
  const rsrc_t zres = make_rsrc(a.zeros, (uint32_t)a.qrows * (N >> 3) * 4u);
  const rsrc_t xres = make_rsrc(a.x, (uint32_t)a.M * K * 2u);
  const uint32_t wlane = (uint32_t)(t0 * 64 + lane) * 16u;
  uint32_t xlane[XN];
#pragma unroll
  for (int j = 0; j < XN; ++j) xlane[j] = ((uint32_t)min(4 * j + kq, a.M - 1) * K + 8 * c) * 2u;
  auto load = [&](Block& b, int i) {
    const int g = wave + W * i;
    const uint32_t oob = g < G ? 0u : 0x80000000u;           // past the last block: zeros, no traffic
#pragma unroll
    for (int j = 0; j < XN; ++j) b.x[j] = buf_load16(xres, xlane[j] + (uint32_t)g * 256u + oob);
#pragma unroll
    for (int t = 0; t < NT; ++t) b.w[t] = buf_load16_nt(wres, wlane + (uint32_t)g * 8192u + oob + t * 1024);
    const uint32_t row = a.gpk_magic ? __umulhi((uint32_t)g, a.gpk_magic) : (uint32_t)g;
    load_halves<NT>(sres, (row * N + ncol) * 2u + oob, b.s);
    b.z[0] = 0x88888888u;
    if (ZK == MI355Q_ZP_PACKED) b.z[0] = __builtin_amdgcn_raw_buffer_load_b32(zres, (int)((row * (N >> 3) + (ncol8 >> 3)) * 4u + oob), 0, 0);
  };
  const DecodeConst k = decode_const<DT>();
  // x: written as fetched, a row of 256 bytes per 16 lanes, read as the MFMA wants it; chunk q of row r lies at q ^ r
  unsigned char* const xl = lds + wave * (1024 * XN);
  uint32_t xw[XN], xr[4];
#pragma unroll
  for (int j = 0; j < XN; ++j) xw[j] = (uint32_t)((4 * j + kq) * 256 + (c ^ (4 * j + kq)) * 16);
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    const int r = XN == 4 ? c : c & (4 * XN - 1);      // (rows past the last: any, they are not stored)
    xr[s] = (uint32_t)(r * 256 + ((4 * s + kq) ^ r) * 16);
  }

  f4 acc[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) acc[t] = (f4){0.f, 0.f, 0.f, 0.f};
  auto compute = [&](Block& b) {
    u4 x[4];
#pragma unroll
    for (int j = 0; j < XN; ++j) *(u4*)(xl + xw[j]) = b.x[j];
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int s = 0; s < 4; ++s) x[s] = *(const u4*)(xl + xr[s]);
    __builtin_amdgcn_wave_barrier();
    decode_block<DT, ZK, NT>(acc, x, b, t0, k);
  };
  {
    Block blk[B];
#pragma unroll
    for (int i = 0; i < B; ++i) load(blk[i], i);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < B; ++i) {
      compute(blk[i]);
      __builtin_amdgcn_sched_barrier(0);
    }
  }

  // ---- the wavefronts' sums meet in LDS: wavefront v adds and stores CW of the 4 NT values of a lane
  constexpr int CW = 4 * NT / W > 0 ? 4 * NT / W : 1;
  float (*red)[4 * NT][64] = (float (*)[4 * NT][64])lds;
  __syncthreads();
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) red[wave][i * NT + t][lane] = acc[t][i];
  __syncthreads();
  if (wave * CW >= 4 * NT) return;
  const int q0 = wave * CW, ri = q0 / NT, tc = q0 % NT;
  float fin[CW];
#pragma unroll
  for (int t = 0; t < CW; ++t) {
    float v = red[0][q0 + t][lane];
#pragma unroll
    for (int w = 1; w < W; ++w) v += red[w][q0 + t][lane];
    fin[t] = v;
  }
  const int m = 4 * kq + ri;
  const uint16_t* const bias = a.bias ? a.bias + ncol + tc : nullptr;
  uint16_t* const out = a.out + (size_t)m * N + ncol + tc;
  // (written through to memory: nothing is left for the end of the kernel to write back)
  if (m < a.M) store_row<DT, CW>(out, bias, fin);
}

// ---- grouped (fused-MoE) launches: blocks of 16 slots, decode-sized token counts -------------------------------------------
// Bound by the weights of the experts that have slots, and next to them by the address unit, through which the activations
// come as well: a block with four or eight slots asks for four or eight rows and not for sixteen, 256 bytes of a row at a time (four
// lanes to a row, as the streaming kernel reads them, cost that unit twice as much).  Weights and activations are asked for
// one K block ahead; wavefronts take the K blocks in turn and add their sums through LDS.  128 registers and four wavefronts on a SIMD with
// up to four tiles, two with eight.
// Measured (us for a whole fused-MoE layer, fp16, groups of 128, on the streaming kernel -> here): eight experts of 4096 x 28672 and
// 14336 x 4096, two to a token, at 1 / 4 / 16 / 32 tokens 68.0 / 115.1 / 140.2 / 148.3 -> 51.9 / 106.3 / 134.1 / 142.0; sixty of
// 2048 x 2816 and 1408 x 2048, four to a token, at 1 / 8 / 32 / 64 31.7 / 50.9 / 71.9 / 78.2 -> 31.2 / 44.5 / 64.7 / 73.1; sixteen of
// 3072 x 8192 and 4096 x 3072, two to a token, at 3 / 16 / 48 47.3 / 72.8 / 78.2 -> 42.9 / 68.6 / 78.0.
// IDS: up to 64 slots, given by their experts and not sorted: every wavefront finds the workgroup's block by itself -- the slots of an
// expert from ballots of the bits of its number, experts in the order of their first slot, 16 slots to a block -- in less time than
// the loads from a finished alignment take, and the launch that makes one is saved (us for the whole layer as above: eight experts at 1 / 4 /
// 16 / 32 tokens 51.9 / 106.3 / 134.1 / 142.0 -> 47.5 / 101.5 / 129.9 / 138.5, sixty at 8 / 16 44.5 / 55.8 -> 39.3 / 50.3).
// GLU: the columns are gate and up, half of the tiles of a workgroup gate columns and half the up columns that go with them, and what is
// written is silu(gate) * up of the rounded sums, as the operator that follows would: its launch, and half of the stores, are saved (sorted
// blocks, us for a whole layer: 51.0 -> 49.6, 62.8 -> 61.4, 47.0 -> 45.0).
template <int DT, int ZK, int NT, int W, bool IDS, bool GLU>
__global__ void __launch_bounds__(64 * W, NT == 8 ? 2 : 4)
w4a16_decode_grouped_kernel(DecodeArgs a) {
  static_assert(!GLU || (NT >= 4 && ZK != MI355Q_ZP_PRESCALED && W <= 2 * NT), "pairs of tiles, integer zero-points");
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = lane & 15, kq = lane >> 4;
  constexpr int CT = GLU ? NT / 2 : NT, TG = 8 / CT; // tiles in a slab, tile groups of a slab
  const int group = xcd_tile(), slab = group / TG, t0 = (group % TG) * CT;
  const int G = a.K >> 7, N = a.N, K = a.K;
  __shared__ int block_ids[IDS ? 16 : 1];
  const int32_t* const ids = a.sorted_ids + 16 * blockIdx.z;
  auto slot_id = [&](int r) { return IDS ? block_ids[IDS ? r : 0] : ids[r]; };
  long e;
  int real;                                          // slots up to the last that is no pad
  if constexpr (IDS) {
    const SlotBlock b = find_slot_block<4>(a.sorted_ids, a.id_step, a.id_bits, a.numel, a.E, (int)blockIdx.z, lane);
    if (!b.real) return;                             // (as every wavefront of the workgroup)
    e = b.expert;
    real = b.real;
    if (wave == 0) {
      if (lane < 16) block_ids[lane] = a.numel;
      __builtin_amdgcn_wave_barrier();
      if (holds_lane<4>(b)) block_ids[b.rank & 15] = lane;
    }
    __syncthreads();
  } else {
    if (16 * (int)blockIdx.z >= *a.npp) return;
    e = a.expert_ids[blockIdx.z];
    if (e < 0 || e >= a.E) {                         // not one of this rank's experts: zero rows, no weights read
      const float zero[NT] = {};
      const int id = threadIdx.x < 256 ? ids[threadIdx.x >> 4] : a.numel;
      if (id >= a.numel) return;
      if constexpr (GLU) store_row<DT, CT>(a.out + (size_t)id * (N >> 1) + 128 * slab + 8 * c + t0, nullptr, *(const float(*)[CT])zero);
      else store_row<DT, NT>(a.out + (size_t)id * N + 128 * slab + 8 * c + t0, nullptr, zero);
      return;
    }
    real = 64 - __clzll(__ballot(lane < 16 && ids[c] < a.numel));
  }
  const int ncol8 = 128 * slab + 8 * c, ncol = ncol8 + t0;
  constexpr int RED = W * 4 * NT * 64 * 4, XL = W * 4096;
  __shared__ __align__(16) unsigned char lds[RED > XL ? RED : XL];
  typedef DecodeBlock<NT, ZK, GLU> Block;
  const char* const wslab = (const char*)a.qw + e * a.w_stride + (size_t)slab * G * 8192;
  const rsrc_t wres = make_rsrc(wslab, (uint32_t)G * 8192u), upres = make_rsrc(wslab + (GLU ? (size_t)(N >> 8) * G * 8192 : 0), (uint32_t)G * 8192u);
  const rsrc_t sres = make_rsrc((const char*)a.scales + e * a.s_stride, (uint32_t)a.qrows * N * 2u);
  const rsrc_t zres = make_rsrc(ZK == MI355Q_ZP_NONE ? nullptr : (const char*)a.zeros + e * a.z_stride,
                                (uint32_t)a.qrows * (ZK == MI355Q_ZP_PRESCALED ? N * 2u : (N >> 1)));
  const rsrc_t xres = make_rsrc(a.x, (uint32_t)a.M * K * 2u);
  const uint32_t wlane = (uint32_t)(t0 * 64 + lane) * 16u;
  const int g0 = (int)blockIdx.y * a.kper + wave, nb = (min(G - (int)blockIdx.y * a.kper, a.kper) - wave + W - 1) / W;
  auto load = [&](Block& b, int i) {
    const int g = g0 + W * min(i, nb);
    const uint32_t oob = i < nb ? 0u : 0x80000000u;            // past the last block: zeros, no traffic
#pragma unroll
    for (int t = 0; t < NT; ++t) b.w[t] = buf_load16_nt(GLU && t >= CT ? upres : wres, wlane + (uint32_t)g * 8192u + oob + (t % CT) * 1024);
    const uint32_t row = a.gpk_magic ? __umulhi((uint32_t)g, a.gpk_magic) : (uint32_t)g;
    load_halves<CT>(sres, (row * N + ncol) * 2u + oob, b.s);
    if constexpr (GLU) load_halves<CT>(sres, (row * N + (N >> 1) + ncol) * 2u + oob, b.s + CT / 2);
    b.z[0] = 0x88888888u;
    if constexpr (GLU) b.z[1] = ZK == MI355Q_ZP_PACKED ? __builtin_amdgcn_raw_buffer_load_b32(zres, (int)((row * (N >> 3) + ((ncol8 + (N >> 1)) >> 3)) * 4u + oob), 0, 0) : 0x88888888u;
    if constexpr (ZK == MI355Q_ZP_PACKED) b.z[0] = __builtin_amdgcn_raw_buffer_load_b32(zres, (int)((row * (N >> 3) + (ncol8 >> 3)) * 4u + oob), 0, 0);
    if constexpr (ZK == MI355Q_ZP_PRESCALED) load_halves<NT>(zres, (row * N + ncol) * 2u + oob, b.z);
  };
  const DecodeConst k = decode_const<DT>();
  unsigned char* const xl = lds + wave * 4096;
  uint32_t xw[4], xr[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    xw[j] = (uint32_t)((4 * j + kq) * 256 + (c ^ (4 * j + kq)) * 16);
    xr[j] = (uint32_t)(c * 256 + ((4 * j + kq) ^ c) * 16);
  }
  f4 acc[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) acc[t] = (f4){0.f, 0.f, 0.f, 0.f};
  // the K blocks of this wavefront with 4 XN rows of activations: weights one block ahead of the arithmetic, activations too
  auto run = [&](auto rows) __attribute__((always_inline)) {
    constexpr int XN = decltype(rows)::value;
    uint32_t xlane[XN];
#pragma unroll
    for (int j = 0; j < XN; ++j) xlane[j] = ((uint32_t)(min(slot_id(4 * j + kq), a.numel - 1) / a.topk) * (uint32_t)K + 8u * c) * 2u;   // (pads read a valid row)
    u4 xv[XN];
    auto load_x = [&](int i) {
      const uint32_t at = (uint32_t)(g0 + W * min(i, nb)) * 256u + (i < nb ? 0u : 0x80000000u);
#pragma unroll
      for (int j = 0; j < XN; ++j) xv[j] = buf_load16(xres, xlane[j] + at);
    };
    Block ring[2];
    auto step = [&](const Block& cur, Block& nxt, int i) __attribute__((always_inline)) {
#pragma unroll
      for (int j = 0; j < XN; ++j) *(u4*)(xl + xw[j]) = xv[j];
      __builtin_amdgcn_wave_barrier();
      load_x(i + 1);
      load(nxt, i + 1);
      __builtin_amdgcn_sched_barrier(0);
      u4 x[4];
#pragma unroll
      for (int s = 0; s < 4; ++s) x[s] = *(const u4*)(xl + xr[s]);
      __builtin_amdgcn_wave_barrier();
      decode_block<DT, ZK, NT, GLU>(acc, x, cur, t0, k);
      __builtin_amdgcn_sched_barrier(0);
    };
    load_x(0);
    load(ring[0], 0);
    for (int i = 0;;) {
      step(ring[0], ring[1], i);
      if (++i >= nb) break;
      step(ring[1], ring[0], i);
      if (++i >= nb) break;
    }
  };
  if (nb > 0) {
    if (real <= 4) run(std::integral_constant<int, 1>());
    else if (real <= 8) run(std::integral_constant<int, 2>());
    else run(std::integral_constant<int, 4>());
  }

  constexpr int CW = 4 * NT / W > 0 ? 4 * NT / W : 1;
  float (*red)[4 * NT][64] = (float (*)[4 * NT][64])lds;
  __syncthreads();
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) red[wave][i * NT + t][lane] = acc[t][i];
  __syncthreads();
  if constexpr (GLU) {
    constexpr int CP = 4 * CT / W;                     // pairs of a wavefront
    const int p0 = wave * CP, ri = p0 / CT, tc = p0 % CT;
    const int id = slot_id(4 * kq + ri);
    if (id >= a.numel) return;
    float fin[CP];
#pragma unroll
    for (int t = 0; t < CP; ++t) {
      const int g = ri * NT + tc + t, u = g + CT;
      float vg = red[0][g][lane], vu = red[0][u][lane];
#pragma unroll
      for (int w = 1; w < W; ++w) vg += red[w][g][lane], vu += red[w][u][lane];
      fin[t] = Elem<DT>::to_f32(silu_mul16<DT>(Elem<DT>::from_f32(vg), Elem<DT>::from_f32(vu)));
    }
    store_row<DT, CP>(a.out + (size_t)id * (N >> 1) + ncol + tc, nullptr, fin);
    return;
  }
  if (wave * CW >= 4 * NT) return;
  const int q0 = wave * CW, ri = q0 / NT, tc = q0 % NT;
  const int id = slot_id(4 * kq + ri);
  if (id >= a.numel) return;
  float fin[CW];
#pragma unroll
  for (int t = 0; t < CW; ++t) {
    float v = red[0][q0 + t][lane];
#pragma unroll
    for (int w = 1; w < W; ++w) v += red[w][q0 + t][lane];
    fin[t] = v;
  }
  if (a.partial) {
    float* const p = a.partial + ((size_t)blockIdx.y * a.numel + id) * N + ncol + tc;
    if constexpr (CW % 4 == 0) {
#pragma unroll
      for (int t = 0; t < CW; t += 4) *(f4*)(p + t) = (f4){fin[t], fin[t + 1], fin[t + 2], fin[t + 3]};
    } else {
#pragma unroll
      for (int t = 0; t < CW; ++t) p[t] = fin[t];
    }
    return;
  }
  if (a.topk_weights) {
    const float rw = a.topk_weights[id];
#pragma unroll
    for (int t = 0; t < CW; ++t) fin[t] *= rw;
  }
  store_row<DT, CW>(a.out + (size_t)id * N + ncol + tc, nullptr, fin);
}

template <int DT, int ZK, int NT, int W, int B, int XN>
void launch(const DecodeArgs& a, hipStream_t st) {
  hipLaunchKernelGGL((w4a16_decode_kernel<DT, ZK, NT, W, B, XN>), dim3(a.N / 128 * (8 / NT)), dim3(64 * W), 0, st, a);
}

// tiles of 16 columns per workgroup, wavefronts, K blocks of a wavefront; nt 0: not a problem for this kernel
struct DecodePlan {
  int nt, w, b;
};
DecodePlan decode_plan(int M, int K, int N) {
  const int G = K / 128, cus = device_cu_count();
  if (M > 16 || G > (M > 8 ? 32 : 112)) return {0, 0, 0};
  int nt = 1;
  while (nt <= 4 && N / 16 / nt > cus) nt *= 2;
  if (nt > (M > 8 ? 2 : 4) || (nt == 4 && G > 48)) return {0, 0, 0};
  // Deep K: as many K blocks of a wavefront as its registers hold, where most CUs have a tile.  (us, the streaming kernel with its exchange
  // between K ranges -> here, fp16, at 1 / 4 rows: 8704 x 4096 8.1 / 8.7 -> 7.1 / 7.2, 14336 x 4096 10.2 / 10.7 -> 9.7 / 9.6, 10240 x 8192
  // 12.8 / 12.2 -> 11.3 / 11.2, 8704 x 2048 7.0 / 7.5 -> 6.3 / 6.7; at 8 rows 8704 x 4096 8.7 -> 8.3.  Behind: 16384 x 8192 at 1 16.5 / 23, 13824 x 5120 11.1 /
  // 13.4, both beyond the registers, 14336 x 4096 at 8 10.6 / 11.1, 8704 x 2048 at 8, bf16, 7.4 / 8.0; 14336 x 2048 at 2, bf16, 8.2 / 8.2.)
  const int wgs = N / 16 / nt;
  if (G > 64 && (nt == 4 || 2 * wgs < cus || G > (M > 4 || nt == 2 ? 80 : 4 * wgs < 3 * cus ? 96 : 112) || (M > 4 && 4 * wgs < 3 * cus))) return {0, 0, 0};
  const int w = G <= 16 || (G <= 32 && M <= 8 && nt <= 2) ? 8 : 16;
  return {nt, w, (G + w - 1) / w};
}

template <int DT, int ZK, int NT>
void launch_plan(const DecodePlan& p, const DecodeArgs& a, hipStream_t st) {
#define MQ_D(W, B, XN) if (p.w == W && p.b == B && a.M <= 4 * XN) return launch<DT, ZK, NT, W, B, XN>(a, st)
  MQ_D(8, 1, 1); MQ_D(8, 2, 1); MQ_D(16, 3, 1);
  MQ_D(8, 1, 2); MQ_D(8, 2, 2); MQ_D(16, 3, 2);
  if constexpr (NT <= 2) {
    MQ_D(8, 3, 1); MQ_D(8, 4, 1); MQ_D(16, 4, 1);
    MQ_D(8, 3, 2); MQ_D(8, 4, 2); MQ_D(16, 4, 2);
    MQ_D(8, 1, 4); MQ_D(8, 2, 4); MQ_D(16, 2, 4);
    MQ_D(16, 5, 1); MQ_D(16, 5, 2);
    if constexpr (NT == 1) {
      MQ_D(16, 6, 1); MQ_D(16, 7, 1);
    }
  } else {
    MQ_D(16, 2, 1); MQ_D(16, 2, 2);
  }
#undef MQ_D
}

}  // namespace

// Whether this kernel is the one to take: as few tiles of 16 columns per workgroup as one round of workgroups allows, K within
// what the wavefronts hold.  Above it the streaming kernel is ahead (us, it / here: 4096 x 12288 at 16 rows 8.5 / 8.9, 5120 x 5120 at 16
// 7.5 / 8.2, 4096 x 28672 at 1 12.0 / 12.7, 14336 x 4096 at 16 in four ranges 10.6 / 11.9); pre-scaled zero-points and groups below 128
// stay with it as well.
bool w4a16_decode_wanted(int M, int K, int N, int group_size, int zeros_kind) {
  return group_size % 128 == 0 && zeros_kind != MI355Q_ZP_PRESCALED && (size_t)(K / group_size) * N * 2 < ((size_t)1 << 31) &&
         decode_plan(M, K, N).nt > 0;
}

// (a shape that w4a16_decode_wanted takes; no workspace)
int w4a16_decode_launch(void* out, const void* x, const int32_t* qweight, const void* scales, const void* zeros, int zeros_kind,
                        const void* bias, int M, int K, int N, int group_size, int dtype, hipStream_t st) {
  const DecodePlan p = decode_plan(M, K, N);
  DecodeArgs a = {};
  a.out = (uint16_t*)out; a.x = (const uint16_t*)x; a.qw = (const u4*)qweight; a.scales = (const uint16_t*)scales; a.zeros = zeros;
  a.bias = (const uint16_t*)bias;
  a.M = M; a.K = K; a.N = N;
  const uint32_t gpk = (uint32_t)group_size / 128u;
  a.gpk_magic = gpk > 1 ? (uint32_t)((((uint64_t)1 << 32) + gpk - 1) / gpk) : 0u;
  a.qrows = K / group_size;
#define MQ_NT(DT, ZK)                                            \
  do {                                                           \
    if (p.nt == 1) launch_plan<DT, ZK, 1>(p, a, st);             \
    else if (p.nt == 2) launch_plan<DT, ZK, 2>(p, a, st);        \
    else launch_plan<DT, ZK, 4>(p, a, st);                       \
  } while (0)
  if (dtype == MI355Q_F16 && zeros_kind == MI355Q_ZP_PACKED) MQ_NT(MI355Q_F16, MI355Q_ZP_PACKED);
  else if (dtype == MI355Q_F16) MQ_NT(MI355Q_F16, MI355Q_ZP_NONE);
  else if (zeros_kind == MI355Q_ZP_PACKED) MQ_NT(MI355Q_BF16, MI355Q_ZP_PACKED);
  else MQ_NT(MI355Q_BF16, MI355Q_ZP_NONE);
#undef MQ_NT
  MQ_LAUNCH_CHECK("w4a16_gemm(decode)");
  return 0;
}

namespace {
// Tiles of 16 columns per workgroup and its wavefronts, by the 128-column slabs of weights that the launch is expected to read.  (Which
// blocks hold slots is known on the device only; here, how many experts evenly spread slots reach.)  Fewer slabs than a
// third of the CUs: a CU each for the quarters of a slab, and all its wavefronts (second GEMM of one token of eight experts, 64 slabs:
// the layer 53.6 us with two tiles and eight wavefronts, 56.7 with four and eight, 59.3 with four and four).  Up to the CUs: half
// slabs (3 tokens, 160 slabs: 98 against 105 with quarters).  About the CUs: whole ones, eight wavefronts (16 tokens, 256 slabs: 129 against
// 130 with halves, and at 32 tokens 143 against 149).  Beyond that the rows decide: a half slab reads the activations twice
// for a slab, which few rows make up with four wavefronts on a SIMD and many don't (first GEMM at 3 tokens 98 with halves, 100 whole;
// at 32 tokens 170 and 149; sixty experts of 2048 x 2816, 64 tokens: 85 and 73).
struct GroupedPlan {
  int nt, w;
};
GroupedPlan grouped_plan(int numel, int max_blocks, int E, int N) {
  const double hit = E * (1.0 - std::pow(1.0 - 1.0 / E, numel)), slabs = N / 128 * std::min(hit, (double)max_blocks), cus = device_cu_count();
  if (slabs < 0.33 * cus) return {2, 8};
  if (slabs < 0.8 * cus) return {4, 4};
  if (slabs < 1.05 * cus) return {8, 8};
  if (slabs < (numel < 3 * hit ? 6 : numel < 7 * hit ? 2.2 : 0) * cus) return {4, 4};
  return {8, 4};
}

// K ranges of the second GEMM.  Quarters of a slab with fewer than three workgroups per CU leave CUs with one more than others, and a CU
// takes no more than its 25 GB/s from memory: half or a quarter of K each, their sums added by the launch that adds the slots, even that out.  (us
// for the layer, fp16, 1 / 2 / 4 ranges; eight experts of 4096 x 28672 and 14336 x 4096 at 2 / 3 / 5 tokens, 211 / 282 / 378 workgroups 80.7 / 97.7 /
// 104.2, 77.8 / 96.2 / 100.6, 78.6 / 92.4 / 100.5; sixteen of 3072 x 12288 and 6144 x 3072 at 4 / 16 / 32 51.2 / 85.2 / 95.4, 50.8 / 82.9 / 95.0,
// 49.3 / 83.6 / 96.2; bf16 by the same lines.  Whole slabs and short K lose: eight experts at 16 tokens 136 / 141 / 145, sixty of 1408 x 2048 at 4 31.3 / 34.4 / 36.1.)
int sum_ranges(int numel, int E, int K, int N) {
  const GroupedPlan p = grouped_plan(numel, std::min(numel, (numel + E * 15) / 16), E, N);
  if (p.nt != 4) return 1;
  const long cus = device_cu_count();
  const double wgs = N / 64 * E * (1.0 - std::pow(1.0 - 1.0 / E, numel));
  const int s = wgs > 3 * cus ? 1 : wgs > 2 * cus || wgs <= cus ? 2 : 4;
  return std::min(s, K / 128 >= 48 ? 4 : K / 128 >= 24 ? 2 : 1);
}

// out[m, n] = sum over a token's slots of the slot's sum over the K ranges times its routing weight, rounded to the output type as
// the grouped GEMM and moe_sum round it one after the other.  (Bound by its launch; f32 sums from the GEMM cost nothing next to rounded ones:
// eight experts of 4096 x 14336 at 16 / 32 tokens, one range, 139 / 146 -> 136 / 142 us for the layer; at 256 / 512, where blocks of 64 slots have
// K ranges and each had a launch of its own for their sums, 331 / 506 -> 327 / 501.  With the ids read and two slots on their way at a time 9.8 us
// for three ranges of 1024 slots x 4096, 9.3 without either.)
// row_scale: of bf16 rows staged as fp16, or null.  ids: the slots' experts, id_step words apart: a slot of an id outside [0, E) is in no block,
// nobody wrote its sums, and it adds nothing.
template <int DT, int S>
__global__ void __launch_bounds__(256)
moe_range_sum_kernel(uint16_t* out, const float* partial, const float* topk_weights, const float* row_scale, const int32_t* ids, int id_step, uint32_t E,
                     uint32_t rows, int T, FastDiv quads) {
  const uint32_t q = blockIdx.x * 256 + threadIdx.x;
  if (q >= rows * quads.d) return;
  const uint32_t m = quads.div(q), n = q - m * quads.d;
  const size_t step = (size_t)rows * T * quads.d;
  f4 acc = {0.f, 0.f, 0.f, 0.f};
  for (int t = 0; t < T; t += 2) {                     // two slots on their way at a time
    f4 v[2][S];
    float rw[2], rs[2];
    uint32_t keep[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const uint32_t slot = m * T + min(t + u, T - 1);
      const f4* const p = (const f4*)partial + (size_t)slot * quads.d + n;
#pragma unroll
      for (int r = 0; r < S; ++r) v[u][r] = p[r * step];
      rw[u] = topk_weights[slot];
      rs[u] = row_scale ? row_scale[slot] : 1.f;
      const uint32_t mask = slot_mask(ids[slot * id_step], E);
      keep[u] = t + u < T ? mask : 0u;
    }
#pragma unroll
    for (int u = 0; u < 2; ++u) {
#pragma unroll
      for (int r = 1; r < S; ++r) v[u][0] += v[u][r];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float p = v[u][0][e] * rw[u];
        if (row_scale) p *= rs[u];
        asm volatile("" : "+v"(p));                    // (a product of its own, as the GEMM's: not one that is rounded to 16 bits at once)
        acc[e] += bitcast<float>(bitcast<uint32_t>(Elem<DT>::to_f32(Elem<DT>::from_f32(p))) & keep[u]);
      }
    }
  }
  u2 o;
  o.x = (uint32_t)Elem<DT>::from_f32(acc[0]) | ((uint32_t)Elem<DT>::from_f32(acc[1]) << 16);
  o.y = (uint32_t)Elem<DT>::from_f32(acc[2]) | ((uint32_t)Elem<DT>::from_f32(acc[3]) << 16);
  ((u2*)out)[q] = o;
}

template <int DT, int ZK, bool IDS, bool GLU = false>
void launch_grouped(const DecodeArgs& a, GroupedPlan p, int blocks, hipStream_t st) {
  const int ranges = (a.K / 128 + a.kper - 1) / a.kper;
#define MQ_G(NT, W) \
  if (p.nt == NT && p.w == W) hipLaunchKernelGGL((w4a16_decode_grouped_kernel<DT, ZK, NT, W, IDS, GLU>), dim3(a.N / 128 * (8 / NT), ranges, blocks), dim3(64 * W), 0, st, a)
  MQ_G(8, 4); MQ_G(8, 8); MQ_G(4, 4);
  if constexpr (GLU) {
    MQ_G(4, 8);
  } else {
    MQ_G(2, 8);
  }
#undef MQ_G
}
}  // namespace

// expert_ids null: sorted_ids are the experts of the slots themselves, id_step words apart.  glu: out [numel, N / 2] (packed zero-points or none)
int w4a16_decode_grouped_launch(void* out, const void* x, const int32_t* qweight, const void* scales, const void* zeros, int zeros_kind,
                                const float* topk_weights, const int32_t* sorted_ids, const int32_t* expert_ids, const int32_t* npp,
                                int numel, int topk, int max_blocks, int E, int K, int N, int group_size, int dtype, hipStream_t st, int id_step = 1, bool glu = false,
                                int kper = 0, float* partial = nullptr) {
  MQ_REQUIRE(group_size % 128 == 0 && K % 128 == 0 && N % 128 == 0,
             "moe_w4a16(decode): K=%d, N=%d and group_size=%d must be multiples of 128", K, N, group_size);
  const int rows = numel / (topk > 0 ? topk : 1) + 1;
  MQ_REQUIRE((size_t)rows * K * 2 < ((size_t)1 << 31) && (size_t)(K / group_size) * N * 2 < ((size_t)1 << 31) &&
                 (size_t)K * group_size < ((size_t)1 << 32),
             "moe_w4a16(decode): activations and one expert's scales must each stay below 2 GiB (K=%d N=%d)", K, N);
  DecodeArgs a = {};
  a.out = (uint16_t*)out; a.x = (const uint16_t*)x; a.qw = (const u4*)qweight; a.scales = (const uint16_t*)scales; a.zeros = zeros;
  a.M = (numel + topk - 1) / topk;                   // rows of x
  a.K = K; a.N = N;
  const uint32_t gpk = (uint32_t)group_size / 128u;
  a.gpk_magic = gpk > 1 ? (uint32_t)((((uint64_t)1 << 32) + gpk - 1) / gpk) : 0u;
  a.qrows = K / group_size;
  a.sorted_ids = sorted_ids; a.expert_ids = expert_ids; a.npp = npp; a.topk_weights = topk_weights;
  a.numel = numel; a.topk = topk; a.E = E;
  a.id_step = id_step;
  while ((1 << a.id_bits) < E) ++a.id_bits;
  a.w_stride = (long)K * N / 2;
  a.s_stride = (long)(K / group_size) * N * 2;
  a.z_stride = zeros_kind == MI355Q_ZP_PACKED ? (long)(K / group_size) * N / 2 : a.s_stride;
  a.kper = kper > 0 ? kper : K / 128;
  a.partial = partial;
  GroupedPlan p = grouped_plan(numel, max_blocks, E, N);
  if (glu && p.nt == 2) p.nt = 4;                    // (pairs of tiles)
#define MQ_IDS(DT, ZK)                                                       \
  do {                                                                       \
    constexpr int Z = ZK == MI355Q_ZP_PRESCALED ? MI355Q_ZP_NONE : ZK;       \
    if (ZK == Z && glu && expert_ids) launch_grouped<DT, Z, false, true>(a, p, max_blocks, st);  \
    else if (ZK == Z && glu) launch_grouped<DT, Z, true, true>(a, p, max_blocks, st);            \
    else if (expert_ids) launch_grouped<DT, ZK, false>(a, p, max_blocks, st); \
    else launch_grouped<DT, ZK, true>(a, p, max_blocks, st);                 \
  } while (0)
#define MQ_ZK(DT)                                                                      \
  do {                                                                                 \
    if (zeros_kind == MI355Q_ZP_NONE) MQ_IDS(DT, MI355Q_ZP_NONE);                      \
    else if (zeros_kind == MI355Q_ZP_PACKED) MQ_IDS(DT, MI355Q_ZP_PACKED);             \
    else MQ_IDS(DT, MI355Q_ZP_PRESCALED);                                              \
  } while (0)
  if (dtype == MI355Q_F16) MQ_ZK(MI355Q_F16);
  else MQ_ZK(MI355Q_BF16);
#undef MQ_ZK
#undef MQ_IDS
  MQ_LAUNCH_CHECK("moe_w4a16(decode)");
  return 0;
}

// out [rows, N] from f32 sums [ranges][rows * topk][N]; up to six ranges
int moe_range_sum_launch(void* out, const float* partial, const float* topk_weights, const float* row_scale, const int32_t* ids, int id_step, int E, int rows,
                         int topk, int N, int ranges, int dtype, hipStream_t st) {
  const FastDiv quads((uint32_t)(N / 4));
  const dim3 grid((unsigned)(((size_t)rows * (N / 4) + 255) / 256));
#define MQ_S(DT, S) \
  if (ranges == S) hipLaunchKernelGGL((moe_range_sum_kernel<DT, S>), grid, dim3(256), 0, st, (uint16_t*)out, partial, topk_weights, row_scale, ids, id_step, (uint32_t)E, \
                                       (uint32_t)rows, topk, quads)
#define MQ_DT(DT)                                                             \
  do {                                                                        \
    MQ_S(DT, 1); MQ_S(DT, 2); MQ_S(DT, 3); MQ_S(DT, 4); MQ_S(DT, 5); MQ_S(DT, 6); \
  } while (0)
  if (dtype == MI355Q_F16) MQ_DT(MI355Q_F16);
  else MQ_DT(MI355Q_BF16);
#undef MQ_DT
#undef MQ_S
  MQ_LAUNCH_CHECK("moe sum of K ranges");
  return 0;
}

}  // namespace mi355q

using namespace mi355q;

extern "C" int mi355q_w4a16_decode_plan(int M, int K, int N, int* tiles, int* wavefronts, int* k_blocks) {
  MQ_REQUIRE(M > 0 && K > 0 && N > 0 && K % 128 == 0 && N % 128 == 0, "w4a16_decode_plan: bad shape M=%d K=%d N=%d", M, K, N);
  MQ_REQUIRE(tiles && wavefronts && k_blocks, "w4a16_decode_plan: null pointer");
  const DecodePlan p = decode_plan(M, K, N);
  *tiles = p.nt;
  *wavefronts = p.w;
  *k_blocks = p.b;
  return 0;
}

extern "C" int mi355q_moe_w4a16_unsorted(void* out, const void* a, const int32_t* w, const void* w_scale, const void* w_zeros, int zeros_kind,
                                         int group_size, const float* topk_weights, const void* topk_ids, int ids_are_int64, int numel,
                                         int topk, int E, int K, int N, int silu_and_mul, int dtype, void* stream) {
  MQ_REQUIRE(numel >= 0 && numel <= 64 && topk > 0 && E > 0 && K > 0 && N > 0, "moe_w4a16_unsorted: bad shape numel=%d topk=%d E=%d K=%d N=%d", numel,
             topk, E, K, N);
  if (numel == 0) return 0;
  MQ_REQUIRE(out && a && w && w_scale && topk_ids, "moe_w4a16_unsorted: null pointer");
  MQ_REQUIRE(zeros_kind >= MI355Q_ZP_NONE && zeros_kind <= MI355Q_ZP_PRESCALED && (zeros_kind == MI355Q_ZP_NONE || w_zeros),
             "moe_w4a16_unsorted: zeros_kind %d", zeros_kind);
  MQ_REQUIRE(dtype == MI355Q_F16 || dtype == MI355Q_BF16, "moe_w4a16_unsorted: dtype %d", dtype);
  MQ_REQUIRE(group_size > 0 && K % group_size == 0 && (size_t)N * K < ((size_t)1 << 31), "moe_w4a16_unsorted: group_size=%d K=%d N=%d", group_size, K, N);
  MQ_REQUIRE(!silu_and_mul || (N % 256 == 0 && zeros_kind != MI355Q_ZP_PRESCALED && !topk_weights),
             "moe_w4a16_unsorted: SiLU of gate and up takes N=%d in two halves of whole slabs, zero-points that are not pre-scaled and no routing weights", N);
  return w4a16_decode_grouped_launch(out, a, w, w_scale, w_zeros, zeros_kind, topk_weights, (const int32_t*)topk_ids, nullptr, nullptr, numel, topk,
                                     std::min(numel, (numel + E * 15) / 16), E, K, N, group_size, dtype, as_stream(stream), ids_are_int64 ? 2 : 1, silu_and_mul != 0);
}

extern "C" size_t mi355q_moe_w4a16_unsorted_sum_bytes(int numel, int E, int K, int N) {
  return numel > 0 && E > 0 && K > 0 && N > 0 ? (size_t)sum_ranges(numel, E, K, N) * numel * N * sizeof(float) : 0;
}

extern "C" int mi355q_moe_w4a16_unsorted_sum(void* out, const void* a, const int32_t* w, const void* w_scale, const void* w_zeros, int zeros_kind,
                                             int group_size, const float* topk_weights, const void* topk_ids, int ids_are_int64, int rows, int topk,
                                             int E, int K, int N, int dtype, void* workspace, size_t workspace_bytes, void* stream) {
  MQ_REQUIRE(rows >= 0 && topk > 0 && rows <= 64 / topk && E > 0 && K > 0 && N > 0, "moe_w4a16_unsorted_sum: bad shape rows=%d topk=%d E=%d K=%d N=%d", rows,
             topk, E, K, N);
  if (rows == 0) return 0;
  MQ_REQUIRE(out && a && w && w_scale && topk_ids && topk_weights && workspace, "moe_w4a16_unsorted_sum: null pointer");
  MQ_REQUIRE(zeros_kind >= MI355Q_ZP_NONE && zeros_kind <= MI355Q_ZP_PRESCALED && (zeros_kind == MI355Q_ZP_NONE || w_zeros),
             "moe_w4a16_unsorted_sum: zeros_kind %d", zeros_kind);
  MQ_REQUIRE(dtype == MI355Q_F16 || dtype == MI355Q_BF16, "moe_w4a16_unsorted_sum: dtype %d", dtype);
  MQ_REQUIRE(group_size > 0 && K % group_size == 0 && (size_t)N * K < ((size_t)1 << 31), "moe_w4a16_unsorted_sum: group_size=%d K=%d N=%d", group_size, K, N);
  MQ_REQUIRE(K % 128 == 0 && N % 128 == 0 && group_size % 128 == 0, "moe_w4a16_unsorted_sum: K=%d, N=%d and group_size=%d must be multiples of 128", K, N,
             group_size);
  const int numel = rows * topk, G = K / 128;
  const int s = sum_ranges(numel, E, K, N);
  MQ_REQUIRE(workspace_bytes >= (size_t)s * numel * N * sizeof(float), "moe_w4a16_unsorted_sum: workspace of %zu bytes", workspace_bytes);
  const int kper = (G + s - 1) / s;
  MQ_REQUIRE((G + kper - 1) / kper == s, "moe_w4a16_unsorted_sum: %d K blocks in %d ranges", G, s);
  hipStream_t st = as_stream(stream);
  const int rc = w4a16_decode_grouped_launch(nullptr, a, w, w_scale, w_zeros, zeros_kind, nullptr, (const int32_t*)topk_ids, nullptr, nullptr, numel, 1,
                                             std::min(numel, (numel + E * 15) / 16), E, K, N, group_size, dtype, st, ids_are_int64 ? 2 : 1, false, kper,
                                             (float*)workspace);
  if (rc) return rc;
  return moe_range_sum_launch(out, (const float*)workspace, topk_weights, nullptr, (const int32_t*)topk_ids, ids_are_int64 ? 2 : 1, E, rows, topk, N, s, dtype, st);
}
