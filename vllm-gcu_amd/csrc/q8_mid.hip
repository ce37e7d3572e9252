// 8-bit GEMM on MFMA tiles for a few dozen to some hundred rows: fp8 with 128 x 128 block scales, fp8 with per-token x
// per-channel scales, and int8 (weights in the kslab order).
//
// Between the weight streamer (up to about 32 rows) and the 256 x 128 tiles of the prefill kernels a layer of a few
// thousand columns is neither: the weights are read about once, so HBM is the roof, but every 256-row tile has
// wavefronts without rows, and the few tiles there are walk K at about 1 us per K block (sixteen MFMAs, as many
// operand reads and sixty-four scale multiply-adds in a row per wavefront).  Here a workgroup of four wavefronts owns
// a tile of 32 x 64 or 64 x 64, and two or three workgroups share a CU and fill each other's barrier and LDS waits (or
// eight wavefronts own 128 x 128 rows, alone on it), so that every wavefront has rows and K is cut into fewer ranges,
// there being two to eight times as many tiles.
//
// Every operand travels from global memory straight into a ring of LDS stages (one K block of 128 bytes per row each),
// issued from inline assembly so that the compiler, which does not see the copies, waits for the LDS reads alone; the
// waits for the copies are written by hand.  Activation scales of the whole K range are copied in front, laid out one
// row after the other with an odd pitch.  kslab weights are the LDS image already: a copy is one contiguous KiB.
//
// Measured against the streamer / the 256-row tiles (us): fp8 block 2048 x 7168 at 48 / 128 / 256 / 512 rows 9.1 / 18.6 / 25.6 /
// 26.7 -> 6.4 / 8.0 / 10.2 / 15.6, 7168 x 4096 17.6 / 21.9 / 28.9 / 36.3 -> 11.4 / 15.6 / 20.5 / 30.1; int8 3584 x 4608 16.1 /
// 18.6 / 25.3 / 29.4 -> 7.7 / 9.6 / 13.9 / 21.3, 8192 x 8192 at 128 / 512: 26.0 / 51.8 -> 24.3 / 43.7.  What bounds it: HBM up to
// about 100 rows on large layers; the launch and the filling of the ring (4 us) on small ones; above, the step of a K block
// (0.6 us for 128 x 128 with eight wavefronts: barrier, 12 operand reads, 4 copies and 8 .. 16 matrix instructions each --
// taking out any one of the three saves a fifth), which is why the 256-row tiles win again from about 1000 rows.
#include "common.h"

#include <algorithm>
#include <cmath>
#include <type_traits>

namespace mi355q {

// K ranges of the 256-row tile kernels (1: none), and the int8 one's rounds in units of a round of 256 x 128 tiles
int fp8_ksplits(int M, int N, int K);
double f8_block_rounds(int M, int N, int bm);
int int8_ksplits(int M, int N, int K);
int int8_ksplits_wide(int M, int N, int K);
double int8_tile_rounds(int M, int N);

namespace {

enum { Q8_BLOCK = 0, Q8_PC = 1, Q8_INT8 = 2 };

struct Q8Args {
  void* out;                // [M, N], row stride ldo elements
  const uint8_t* x;         // [M, K], row stride ldx bytes
  const uint8_t* w;         // kslab order
  const float* x_scale;     // block: [M, K / 128]; else [M] or one value, or null (int8)
  const float* w_scale;     // block: [N / 128, K / 128]; else [N] or one value, or null (int8)
  const void* bias;         // [N] in the output dtype, or f32, or null
  int xs_mul, ws_mul, bias_f32;
  int M, N, K;
  long ldx, ldo;
  int kper;                 // K blocks per range (blockIdx.y)
  int mtiles;
  int xcds;                 // the column tiles are a multiple of the eight XCDs
  void* partial;            // split K: f32 / int32 sums [range][M][N]; null: write the output
};

__device__ __forceinline__ void q8_dma16(uint32_t voff, const void* sbase, uint32_t lds_addr) {
  lds_addr = __builtin_amdgcn_readfirstlane(lds_addr);
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"(voff), "s"(sbase), "s"(lds_addr) : "memory");
}
__device__ __forceinline__ void q8_dma4(uint32_t voff, const void* sbase, uint32_t lds_addr) {
  lds_addr = __builtin_amdgcn_readfirstlane(lds_addr);
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dword %0, %1" : : "v"(voff), "s"(sbase), "s"(lds_addr) : "memory");
}
template <int N>
__device__ __forceinline__ void q8_wait_vmcnt() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" : : "n"(N) : "memory");   // (and no LDS read of the stage before is open)
}

typedef int i8v __attribute__((ext_vector_type(8)));

// wavefronts WM x WN, each 16 NJ rows of x by 16 NI rows of w
template <int WM_, int WN_, int NJ_, int NI_, int D_>
struct Q8Cfg {
  static constexpr int WM = WM_, WN = WN_, NJ = NJ_, NI = NI_, D = D_;
  static constexpr int BM = WM * NJ * 16, BN = WN * NI * 16;
  static constexpr int WAVES = WM * WN, THREADS = 64 * WAVES;
  static constexpr int X_BYTES = BM * 128, W_BYTES = BN * 128, STAGE = X_BYTES + W_BYTES;
  static constexpr int XC = X_BYTES / 1024 / WAVES, WC = W_BYTES / 1024 / WAVES, NC = XC + WC;   // copies per wavefront and stage
  static_assert(XC * WAVES * 1024 == X_BYTES && WC * WAVES * 1024 == W_BYTES, "whole copies");
};

template <int DT>
__device__ __forceinline__ float q8_bias(const void* bias, int f32, int n) {
  if (f32 || DT == MI355Q_F32) return ((const float*)bias)[n];
  return Elem<DT == MI355Q_F32 ? MI355Q_F16 : DT>::to_f32(((const uint16_t*)bias)[n]);
}

template <int DT>
__device__ __forceinline__ void q8_store4(void* out, long idx, const float* v) {
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

// (sum * x_scale) * w_scale (+ bias) for 4 adjacent columns, as the other 8-bit kernels do it
template <int MODE, int DT, typename ACC>
__device__ __forceinline__ void q8_finish(const Q8Args& a, int m, int n, const ACC& sum) {
  float v[4];
  const float xs = MODE != Q8_BLOCK && a.x_scale ? a.x_scale[(long)m * a.xs_mul] : 1.0f;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    v[e] = (float)sum[e];
    if (MODE != Q8_BLOCK) v[e] = scaled_sum(v[e], xs, a.w_scale ? a.w_scale[(long)(n + e) * a.ws_mul] : 1.0f);
    if (MODE != Q8_INT8 || a.bias) v[e] = plus_bias(v[e], a.bias ? q8_bias<DT>(a.bias, a.bias_f32, n + e) : 0.0f);
  }
  q8_store4<DT>(a.out, (long)m * a.ldo + n, v);
}

template <int MODE, int DT, typename C>
__global__ void __launch_bounds__(C::THREADS, 2)
q8_mid_kernel(Q8Args a) {
  constexpr int NJ = C::NJ, NI = C::NI, D = C::D, NC = C::NC;
  typedef typename std::conditional<MODE == Q8_INT8, i4, f4>::type acc_t;
  extern __shared__ __align__(16) unsigned char lds[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, kq = lane >> 4;
  const int wm = wave / C::WN, wn = wave % C::WN;
  const int M = a.M, N = a.N, KB = a.K >> 7;
  // consecutive workgroups go to the eight XCDs in turn: the row tiles of a column tile take ids of one residue, so
  // that its weights pass through one L2
  int tm, tn;
  if (a.xcds) {
    const int j = blockIdx.x >> 3;
    tm = j % a.mtiles;
    tn = j / a.mtiles * 8 + (blockIdx.x & 7);
  } else {
    tm = blockIdx.x % a.mtiles;
    tn = blockIdx.x / a.mtiles;
  }
  const int m0 = tm * C::BM, n0 = tn * C::BN;
  const int kb0 = blockIdx.y * a.kper, nk = min(KB - kb0, a.kper);
  const uint32_t lds_base = __builtin_amdgcn_readfirstlane((uint32_t)(size_t)(__attribute__((address_space(3))) unsigned char*)lds);
  const uint32_t scales_off = D * C::STAGE;
  const int pitch = a.kper | 1;                       // floats per row of scales in LDS

  // ---- copies.  x: 8 rows of 128 bytes; lane = 8 * row + position, position p of row r receives chunk p ^ (r & 7)
  uint32_t xo[C::XC];
#pragma unroll
  for (int p = 0; p < C::XC; ++p) {
    const int r = (wave + C::WAVES * p) * 8 + (lane >> 3);
    xo[p] = (uint32_t)(min(m0 + r, M - 1) - m0) * (uint32_t)a.ldx + 16u * (uint32_t)((lane & 7) ^ (r & 7));
  }
  const uint32_t lane16 = (uint32_t)lane * 16u;
  const uint8_t* const xg = a.x + (long)m0 * a.ldx + (long)kb0 * 128;
  // w: KiB c of the tile's K block is KiB c & 7 of 64-row group c >> 3 (kslab: 8 KiB per group and K block)
  const uint8_t* const wg = a.w + ((long)(n0 >> 6) * KB + kb0) * 8192;
  auto copy = [&](int p, int slot, int i) {           // copy p of the NC of a stage
    const int kb = min(i, nk - 1);                    // past the end: a re-read into a stage nobody reads
    const uint32_t sb = lds_base + (uint32_t)(slot * C::STAGE);
    if (p < C::XC) {
      q8_dma16(xo[p < C::XC ? p : 0], xg + (long)kb * 128, sb + (uint32_t)((wave + C::WAVES * p) * 1024));
    } else {
      const int c = wave + C::WAVES * (p - C::XC);
      q8_dma16(lane16, wg + ((long)(c >> 3) * KB + kb) * 8192 + (c & 7) * 1024, sb + (uint32_t)(C::X_BYTES + c * 1024));
    }
  };
  if (MODE == Q8_BLOCK) {
    // scales of the K range: row r of the tile at floats [r * pitch, r * pitch + nk), then the weight scales
    const int total = C::BM * pitch;
    for (int p0 = wave * 64; p0 < total; p0 += C::THREADS) {
      const int p = min(p0 + lane, total - 1), r = p / pitch, kb = min(p - r * pitch, nk - 1);
      q8_dma4((uint32_t)((min(m0 + r, M - 1) - m0) * KB + kb) * 4u, a.x_scale + (long)m0 * KB + kb0,
              lds_base + scales_off + (uint32_t)p0 * 4u);
    }
    const uint32_t ws_off = scales_off + (uint32_t)((total + 63) / 64 * 64) * 4u;
    for (int p0 = wave * 64; p0 < nk; p0 += C::THREADS)
      q8_dma4((uint32_t)min(p0 + lane, nk - 1) * 4u, a.w_scale + (long)(n0 >> 7) * KB + kb0, lds_base + ws_off + (uint32_t)p0 * 4u);
  }
#pragma unroll
  for (int d = 0; d < D; ++d)
#pragma unroll
    for (int p = 0; p < NC; ++p) copy(p, d, d);

  // ---- operand addresses: lane (l16, kq) feeds the MFMA the 16-byte chunks kq and 4 + kq of its row.  (A 16-byte read
  // serves lanes 0-3, 12-15, 20-27 in one pass, 4-11, 16-19, 28-31 in the next: neighbouring kq must lie in chunks of
  // different parity for the swizzle to keep them apart.)
  uint32_t xa[2], wa[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int c = 4 * h + kq;
    xa[h] = (uint32_t)((wm * NJ * 16 + l16) * 128 + ((c ^ (l16 & 7)) * 16));
    wa[h] = (uint32_t)(C::X_BYTES + wn * NI * 2048 + (c & 1) * 1024 + ((c >> 1) * 16 + l16) * 16);
  }
  const float* const xs_l = (const float*)(lds + scales_off) + (wm * NJ * 16 + l16) * pitch;
  const float* const ws_l = (const float*)(lds + scales_off) + (C::BM * pitch + 63) / 64 * 64;

  acc_t acc[NI][NJ];
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) acc[i][j] = (acc_t){0, 0, 0, 0};

  // operands of one K block
  struct Ops {
    i4 w[NI][2], x[NJ][2];
    float xs[NJ], ws;
  };
  auto read_ops = [&](Ops& o, int slot, int i) {
    const unsigned char* st = lds + slot * C::STAGE;
#pragma unroll
    for (int t = 0; t < NI; ++t) {
      o.w[t][0] = *(const i4*)(st + wa[0] + t * 2048);
      o.w[t][1] = *(const i4*)(st + wa[1] + t * 2048);
    }
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      o.x[j][0] = *(const i4*)(st + xa[0] + j * 2048);
      o.x[j][1] = *(const i4*)(st + xa[1] + j * 2048);
    }
    if (MODE == Q8_BLOCK) {
      const int ic = min(i, nk - 1);
#pragma unroll
      for (int j = 0; j < NJ; ++j) o.xs[j] = xs_l[j * 16 * pitch + ic];
      o.ws = ws_l[ic];
    }
  };
  int slot = 0;
  // K block i is multiplied from registers while block i + 1 is read from LDS and block i + D is copied into i's stage
  auto step = [&](const Ops& cur, Ops& nxt, int i) __attribute__((always_inline)) {
    q8_wait_vmcnt<(D - 2) * NC>();                    // this wavefront's copies of block i + 1 have landed, its reads of block i are done
    __builtin_amdgcn_s_barrier();                     // everybody's
    asm volatile("" ::: "memory");
    const int nslot = slot + 1 == D ? 0 : slot + 1;
    read_ops(nxt, nslot, i + 1);
    __builtin_amdgcn_sched_barrier(0);
    // copies between the matrix instructions: the address unit takes 16 .. 20 clocks for each, and a wavefront that
    // issues its copies in a row waits for it with the matrix pipe idle
    constexpr int HV = MODE == Q8_INT8 ? 2 : 1, NM = HV * NI * NJ;      // (int8: the two halves of the K block in turn)
#pragma unroll
    for (int n = 0; n < NM; ++n) {
      const int h = n / (NI * NJ), j = n % (NI * NJ) / NI, t = n % NI;
#pragma unroll
      for (int p = (n * NC + NM - 1) / NM; p < ((n + 1) * NC + NM - 1) / NM; ++p) copy(p, slot, i + D);
      if constexpr (MODE == Q8_INT8) {
        acc[t][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(cur.w[t][h], cur.x[j][h], acc[t][j], 0, 0, 0);
      } else {
        const i8v av = __builtin_shufflevector(cur.w[t][0], cur.w[t][1], 0, 1, 2, 3, 4, 5, 6, 7);
        const i8v bv = __builtin_shufflevector(cur.x[j][0], cur.x[j][1], 0, 1, 2, 3, 4, 5, 6, 7);
        if constexpr (MODE == Q8_PC) {
          acc[t][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(av, bv, acc[t][j], 0, 0, 0, 0, 0, 0);
        } else {
          const f4 part = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(av, bv, (f4){0.f, 0.f, 0.f, 0.f}, 0, 0, 0, 0, 0, 0);
          acc[t][j] += (cur.xs[j] * cur.ws) * part;
        }
      }
      if (MODE != Q8_BLOCK) __builtin_amdgcn_sched_barrier(0);
    }
    slot = nslot;
  };
  Ops o0, o1;
  q8_wait_vmcnt<(D - 1) * NC>();
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  read_ops(o0, 0, 0);
  for (int i = 0;; i += 2) {
    step(o0, o1, i);
    if (i + 1 >= nk) break;
    step(o1, o0, i + 1);
    if (i + 2 >= nk) break;
  }
  q8_wait_vmcnt<0>();                                 // no copy may still be writing LDS when the workgroup retires

  // lane: row m = .. + l16, columns n = .. + 4 kq + {0..3}
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    const int m = m0 + (wm * NJ + j) * 16 + l16;
    if (m >= M) continue;
#pragma unroll
    for (int t = 0; t < NI; ++t) {
      const int n = n0 + (wn * NI + t) * 16 + 4 * kq;
      if (a.partial) *(acc_t*)((acc_t*)a.partial + (((long)blockIdx.y * M + m) * N + n) / 4) = acc[t][j];
      else q8_finish<MODE, DT>(a, m, n, acc[t][j]);
    }
  }
}

// second launch of a split: the ranges' sums in range order, then the epilogue
template <int MODE, int DT>
__global__ void __launch_bounds__(256)
q8_splitk_epilogue_kernel(Q8Args a, int splits, FastDiv quads) {
  typedef typename std::conditional<MODE == Q8_INT8, i4, f4>::type acc_t;
  const uint32_t q = blockIdx.x * 256 + threadIdx.x;
  if (q >= (uint32_t)a.M * quads.d) return;
  const uint32_t m = quads.div(q), nq = q - m * quads.d;
  const acc_t* p = (const acc_t*)a.partial + q;
  const size_t step = (size_t)a.M * quads.d;
  acc_t s = p[0];
  for (int i = 1; i < splits; ++i) s += p[i * step];
  q8_finish<MODE, DT>(a, (int)m, (int)nq * 4, s);
}

typedef Q8Cfg<1, 4, 2, 1, 4> Q8T32;      // 32 x 64, 48 KiB of stages
typedef Q8Cfg<2, 2, 2, 2, 4> Q8T64;      // 64 x 64, 64 KiB
typedef Q8Cfg<2, 4, 4, 2, 4> Q8T128;     // 128 x 128, 128 KiB

template <int MODE, typename C>
size_t q8_lds(int kper) {
  size_t b = (size_t)C::D * C::STAGE;
  if (MODE == Q8_BLOCK) b += ((size_t)(C::BM * (kper | 1) + 63) / 64 * 64 + (kper + 63) / 64 * 64) * sizeof(float);
  return b;
}

template <int MODE, int DT, typename C>
int launch_q8(Q8Args a, int splits, hipStream_t st) {
  const int KB = a.K / 128;
  a.mtiles = (a.M + C::BM - 1) / C::BM;
  a.xcds = (a.N / C::BN) % 8 == 0;
  a.kper = (KB + splits - 1) / splits;
  splits = (KB + a.kper - 1) / a.kper;                // no empty ranges
  if (splits <= 1) a.partial = nullptr;
  const size_t shmem = q8_lds<MODE, C>(a.kper);
  MQ_REQUIRE(shmem <= 160 * 1024, "q8 gemm: %zu bytes of LDS", shmem);
  static hipError_t attr = hipFuncSetAttribute((const void*)q8_mid_kernel<MODE, DT, C>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
  MQ_REQUIRE(attr == hipSuccess, "q8 gemm: cannot reserve LDS: %s", hipGetErrorString(attr));
  hipLaunchKernelGGL((q8_mid_kernel<MODE, DT, C>), dim3((unsigned)(a.mtiles * (a.N / C::BN)), (unsigned)splits), dim3(C::THREADS), shmem, st, a);
  MQ_LAUNCH_CHECK("q8 gemm");
  if (splits > 1) {
    const FastDiv quads((uint32_t)(a.N / 4));
    hipLaunchKernelGGL((q8_splitk_epilogue_kernel<MODE, DT>), dim3((unsigned)(((size_t)a.M * quads.d + 255) / 256)), dim3(256), 0, st, a, splits, quads);
    MQ_LAUNCH_CHECK("q8 gemm (split-K epilogue)");
  }
  return 0;
}

template <int MODE, int DT>
int launch_q8_tile(const Q8Args& a, int bm, int splits, hipStream_t st) {
  if (bm == 32) return launch_q8<MODE, DT, Q8T32>(a, splits, st);
  if (bm == 64) return launch_q8<MODE, DT, Q8T64>(a, splits, st);
  return launch_q8<MODE, DT, Q8T128>(a, splits, st);
}

// ---- which tile, how many K ranges, or which other kernel ---------------------------------------------------
// Prices in us, fitted on MI355X to 13,000 launches: fourteen layers from 1024 x 1024 to 8192 x 28672, 8 .. 1536 rows,
// every tile and 1 .. 16 K ranges, weights rotated past the last-level cache.  A round of workgroups pays a step per K
// block, more of it for every workgroup that shares the CU; the weight stream is a floor; a split pays for its second
// launch and for the bytes of its partial sums.  The pick is within 2 % of the best launch on average.
struct Q8Price {
  double base, split, split_mn;            // launch and ramp; second launch; per million partial sums
  double one[3], more[3];                  // step of one workgroup per CU, of each further one (tiles of 32, 64, 128 rows)
};
constexpr Q8Price kBlockPrice = {3.1, 2.3, 1.29, {0.200, 0.294, 0.973}, {0.185, 0.240, 0.474}};
constexpr Q8Price kPlainPrice = {3.4, 1.6, 1.55, {0.151, 0.232, 0.961}, {0.200, 0.260, 0.190}};
// the 256-row tile kernels: base, step per K block of a round of 256 x 128 tiles, second launch, per million partial sums
struct TilePrice {
  double base, step, split, split_mn;
};
constexpr TilePrice kTilePrice[3] = {{6.5, 0.95, 4.0, 1.61}, {2.6, 0.881, 4.3, 1.70}, {7.2, 0.776, 0.9, 1.83}};

double with_stream(double t, double K, double N) {      // never faster than the weights arrive
  const double h = K * N / 5.05e6;
  return std::sqrt(std::sqrt(t * t * t * t + h * h * h * h));
}

struct Q8Plan {
  int bm, splits;                          // bm 0: another kernel is ahead
  size_t bytes;                            // partial sums
};

double tile_kernel_price(int mode, int M, int N, int K) {
  int splits = mode == Q8_INT8 ? int8_ksplits(M, N, K) : fp8_ksplits(M, N, K);
  const int nk = K / 128;
  const long cus = device_cu_count();
  const TilePrice& p = kTilePrice[mode];
  double rounds = (double)(((long)((M + 255) / 256) * ((N + 127) / 128) * splits + cus - 1) / cus);
  if (mode == Q8_BLOCK && splits == 1) rounds = std::min(f8_block_rounds(M, N, 128), f8_block_rounds(M, N, 256));
  if (mode == Q8_INT8 && splits == 1) {
    const int wide = int8_ksplits_wide(M, N, K);            // ranges of 256 x 256 tiles, one round
    rounds = wide ? 1 / 0.545 : int8_tile_rounds(M, N);
    if (wide) splits = wide;
  }
  double t = p.base + rounds * p.step * nk / splits;
  if (splits > 1) t += p.split + p.split_mn * 1e-6 * splits * M * N;
  return with_stream(t, K, N);
}

Q8Plan q8_make_plan(int mode, int M, int N, int K) {
  Q8Plan best = {0, 1, 0};
  if (M <= 16 || K % 128 != 0 || N % 64 != 0 || (mode == Q8_BLOCK && N % 128 != 0)) return best;
  // The weight streamer stays ahead up to 16 rows, and up to 32 where the weights are large enough for HBM alone to set
  // the pace (us at 32 rows, streamer / here: 8192 x 8192 15.4 / 17.0, 8192 x 28672 44.2 / 48.1, 5120 x 13824 16.2 / 15.4; but
  // 14336 x 4096 19.7 / 15.1, 7168 x 4096 11.4 / 10.9, 3584 x 4608 11.5 / 7.4).
  if (M <= 32 && N >= 8192 && (long)K * N >= (1L << 26)) return best;
  const Q8Price& p = mode == Q8_BLOCK ? kBlockPrice : kPlainPrice;
  const int KB = K / 128;
  const long cus = device_cu_count();
  double least = 1e30;
  for (int c = 0; c < 3; ++c) {
    const int bm = 32 << c, bn = c == 2 ? 128 : 64;
    if (N % bn != 0 || (c > 0 && M <= bm / 2)) continue;
    for (int s = 1; s <= 16; ++s) {
      const int kper = (KB + s - 1) / s, ranges = (KB + kper - 1) / kper;
      if (ranges != s || (s > 1 && kper < 8)) continue;
      const size_t bytes = s > 1 ? (size_t)s * M * N * 4 : 0;
      if (bytes > ((size_t)64 << 20)) continue;
      size_t lds = c == 0 ? q8_lds<Q8_PC, Q8T32>(kper) : c == 1 ? q8_lds<Q8_PC, Q8T64>(kper) : q8_lds<Q8_PC, Q8T128>(kper);
      if (mode == Q8_BLOCK) lds = c == 0 ? q8_lds<Q8_BLOCK, Q8T32>(kper) : c == 1 ? q8_lds<Q8_BLOCK, Q8T64>(kper) : q8_lds<Q8_BLOCK, Q8T128>(kper);
      if (lds > 160 * 1024) continue;
      const long res = std::min<long>(160 * 1024 / lds, 3);
      const long wgs = (long)((M + bm - 1) / bm) * (N / bn) * s, full = wgs / (res * cus), rest = wgs % (res * cus);
      double steps = full * (p.one[c] + p.more[c] * (res - 1));
      if (rest) steps += p.one[c] + p.more[c] * ((rest + cus - 1) / cus - 1);
      double t = with_stream(steps * kper, K, N) + p.base;
      if (s > 1) t += p.split + p.split_mn * 1e-6 * s * M * N;
      if (t < least) {
        least = t;
        best = {bm, s, bytes};
      }
    }
  }
  // the 256-row tiles from 65 rows on (below, half of their wavefronts and more have no rows)
  if (best.bm && M > 64 && N % 128 == 0 && tile_kernel_price(mode, M, N, K) < 1.02 * least) best.bm = 0;
  return best;
}

// (a serving loop asks for the same few shapes again and again, from the host path and from the entry points)
Q8Plan q8_plan(int mode, int M, int N, int K) {
  struct Entry {
    int mode, M, N, K, dev_cus;
    Q8Plan plan;
  };
  static thread_local Entry table[64] = {};
  const uint32_t h = ((uint32_t)M * 2654435761u ^ (uint32_t)N * 40503u ^ (uint32_t)K * 2246822519u ^ (uint32_t)mode) >> 7;
  Entry& e = table[h % 64];
  const int cus = device_cu_count();
  if (e.M != M || e.N != N || e.K != K || e.mode != mode || e.dev_cus != cus) e = {mode, M, N, K, cus, q8_make_plan(mode, M, N, K)};
  return e.plan;
}

}  // namespace

// The plan for a kslab layer: bytes of partial sums, or false where the weight streamer or the 256-row tiles are ahead.
bool q8_mid_wanted(int mode, int M, int N, int K, size_t* bytes) {
  const Q8Plan p = q8_plan(mode, M, N, K);
  *bytes = p.bytes;
  return p.bm != 0;
}

// x_scale / w_scale: block scales (mode 0), or vectors / one value by their index multipliers (0: one value), null = 1 (int8)
int q8_mid_launch(int mode, void* out, const void* x, const void* w, const float* x_scale, int xs_mul, const float* w_scale,
                  int ws_mul, const void* bias, int bias_f32, int M, int N, int K, long ldx, long ldo, int out_dtype, void* partial,
                  hipStream_t st) {
  const Q8Plan p = q8_plan(mode, M, N, K);
  MQ_REQUIRE(p.bm && (p.splits == 1 || partial), "q8 gemm: no plan for M=%d N=%d K=%d", M, N, K);
  Q8Args a = {};
  a.out = out; a.x = (const uint8_t*)x; a.w = (const uint8_t*)w; a.x_scale = x_scale; a.w_scale = w_scale; a.bias = bias;
  a.xs_mul = xs_mul; a.ws_mul = ws_mul; a.bias_f32 = bias_f32;
  a.M = M; a.N = N; a.K = K; a.ldx = ldx; a.ldo = ldo; a.partial = partial;
#define MQ_Q8(MODE)                                                                                       \
  do {                                                                                                    \
    if (out_dtype == MI355Q_F16) return launch_q8_tile<MODE, MI355Q_F16>(a, p.bm, p.splits, st);          \
    if (out_dtype == MI355Q_BF16) return launch_q8_tile<MODE, MI355Q_BF16>(a, p.bm, p.splits, st);        \
    if constexpr (MODE == Q8_INT8) return launch_q8_tile<MODE, MI355Q_F32>(a, p.bm, p.splits, st);        \
    MQ_REQUIRE(false, "q8 gemm: bad out dtype %d", out_dtype);                                            \
  } while (0)
  if (mode == Q8_BLOCK) MQ_Q8(Q8_BLOCK);
  if (mode == Q8_PC) MQ_Q8(Q8_PC);
  MQ_Q8(Q8_INT8);
#undef MQ_Q8
}

}  // namespace mi355q

using namespace mi355q;

extern "C" int mi355q_q8_mid_plan(int kind, int M, int N, int K, size_t* workspace_bytes) {
  size_t bytes = 0;
  const bool yes = M > 0 && N > 0 && K > 0 && kind >= 0 && kind <= 2 && q8_mid_wanted(kind, M, N, K, &bytes);
  if (workspace_bytes) *workspace_bytes = yes && bytes ? ((size_t)1 << 20) + bytes : 0;
  return yes;
}
