// 8-bit GEMM for up to 16 rows, and up to 64 where they are short: fp8 with 128 x 128 block scales, fp8 with per-token x per-channel scales, int8.  Where the rows are few
// thousand elements it takes them as 16-bit values and quantises them itself.
//
// What bounds such a call: HBM on layers of 60 MB and more, and below that what is not overlapped -- the launch, one trip to memory, the sums of the
// wavefronts, and, in front of it all, the launch that quantises the rows (2 .. 3 us on the GPU, 2.5 in the host).  kcontig_gemm_kernel has
// four wavefronts with two K blocks on their way, 16 .. 32 KiB per CU on layers of one or two column tiles per workgroup, and every wavefront
// reads its share of the rows from the L2.  Here one workgroup per CU has eight wavefronts, each with up to eight tiles of 16 columns x one K block on their
// way (128 KiB per CU), requested behind the rows and before anything waits: the rows are quantised, brought into LDS once, in the order the matrix
// operands are read, while the weights arrive.  Rings of 12 and 16 tiles, and 16 wavefronts, were slower everywhere (4096 x 4096 at one row
// 5.5 / 6.0, and 5.6, against 4.7 us): requests past the last K block are not free, which is also why the ring is no longer than a wavefront's share.
//
// Measured (us in a graph, weights out of the caches, int8 with a scale per token; codes: kcontig_gemm_kernel -> here; rows: quantiser and
// kcontig_gemm_kernel -> here): 2048 x 2048 at 1 / 16 rows 3.4 / 4.0 -> 2.9 / 3.1, rows 5.3 -> 3.0; 4096 x 4096 at 1 / 8 5.5 / 5.7 -> 4.7 / 4.8, rows at 1 / 4
// 7.5 / 7.9 -> 4.7 / 6.1; 3584 x 4608 at 16 7.7 -> 5.5; 14336 x 4096 at 1 / 4 13.3 / 12.9 -> 11.2 / 11.1, rows at 1 16.0 -> 12.3; 18944 x 3584 at 1 16.5 -> 13.1, rows
// 19.8 -> 15.3; 8192 x 10240 at 1 / 8 18.7 / 19.1 -> 17.1 / 16.5; 4096 x 28672 at 1 21.7 -> 21.4, rows 23.9 -> 21.4.
// From 17 rows on the weights of a workgroup are multiplied by two, three or four tiles of rows; what it takes is then the copy of the rows, which every
// workgroup makes in whole (the figures stand with the rule, q8_decode_tiles).
#include "q8_few.h"

#include <type_traits>

namespace mi355q {
namespace {

enum { QD_BLOCK = 0, QD_PC = 1, QD_INT8 = 2 };               // as the kinds of q8_mid
enum { QD_CODES = 0, QD_TOKEN = 1, QD_CHANNEL = 2 };         // x: codes; 16-bit rows and a scale per token; ... and a scale per column (int8)

struct QdArgs {
  void* out;                // [M, N] 16 bits
  const void* x;            // [M, K] codes, or 16-bit values in the output's type
  const uint8_t* w;         // [N, K], row-major or in the kslab order
  const float* x_scale;     // QD_CODES: block [M, K / 128]; else [M], one value, or null (1)
  const uint16_t* c_scale;  // QD_CHANNEL: [K] in x's type
  const float* w_scale;     // block [ceil(N / 128), K / 128]; else [N] or one value
  const uint16_t* bias;     // [N] in the output's type, or null
  int sc_row, sc_col;
  int M, N, K, kslab;
  FastDiv row_pieces;       // pieces of 16 bytes in a row of x
};

constexpr int qd_pieces(int src, int waves) { return src == QD_CODES ? 16 : 40 / waves; }   // of x that a thread holds

// NI tiles of 16 columns, W wavefronts, BPR K blocks of each on their way, MT tiles of 16 rows
template <int MODE, int SRC, int DT, int NI, int W, int BPR, int MT>
__global__ void __launch_bounds__(64 * W, 2)
q8_decode_kernel(QdArgs a) {
  static_assert(NI <= W, "the tiles that a wavefront finishes are of the same columns");
  static_assert(SRC == QD_CODES || MODE != QD_BLOCK, "rows for block scales come quantised");
  static_assert(SRC != QD_CHANNEL || MODE == QD_INT8, "scales per column are int8's");
  typedef typename std::conditional<MODE == QD_INT8, i4, f4>::type acc_t;
  constexpr int THREADS = 64 * W, PIECES = qd_pieces(SRC, W);
  extern __shared__ __align__(16) unsigned char lds[];       // x: [K block][row][eight chunks of 16 bytes]; then the wavefronts' sums
  __shared__ uint32_t row_max[16];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15, q = lane >> 4;
  const int M = a.M, N = a.N, K = a.K, KB = K >> 7;
  const int n0 = xcd_tile() * (16 * NI);

  // ---- requests: x, then what the last stores need, then weights (loads return in order, and x is wanted first)
  const int total = M * (int)a.row_pieces.d;
  u4 xv[PIECES], cv[SRC == QD_CHANNEL ? PIECES : 1];
#pragma unroll
  for (int p = 0; p < PIECES; ++p) {
    if (p * THREADS >= total) break;
    const int i = min(tid + p * THREADS, total - 1);
    xv[p] = ((const u4*)a.x)[i];
    if (SRC == QD_CHANNEL) cv[p] = ((const u4*)a.c_scale)[i - (int)(a.row_pieces.div((uint32_t)i) * a.row_pieces.d)];
  }
  if (SRC == QD_TOKEN && tid < 16) row_max[tid] = 0u;
  // tiles wave, wave + W of the NI x MT (columns first): the columns, and the rows, of the outputs that this lane stores
  constexpr int FIN = (NI * MT + W - 1) / W;
  const int nt = n0 + 16 * (wave % NI) + 4 * q;
  const bool stores = wave < NI * MT && nt < N;
  auto stored_row = [&](int f) { return 16 * ((wave + W * f) / NI) + r16; };
  f4 ws = {1.f, 1.f, 1.f, 1.f};
  uint2 bs = {0u, 0u};
  float xs[FIN];
#pragma unroll
  for (int f = 0; f < FIN; ++f) xs[f] = 1.0f;
  if (stores) {
    if (MODE != QD_BLOCK) {
      if (a.sc_col) ws = *(const f4*)(a.w_scale + nt);
      else ws = (f4){a.w_scale[0], a.w_scale[0], a.w_scale[0], a.w_scale[0]};
    }
    if (a.bias) bs = *(const uint2*)(a.bias + nt);
    if (SRC == QD_CODES && MODE != QD_BLOCK && a.x_scale) {
#pragma unroll
      for (int f = 0; f < FIN; ++f) xs[f] = a.x_scale[min(stored_row(f), M - 1) * a.sc_row];
    }
  }
  // block scales of x and of the columns, into LDS behind x: thread t holds values t, t + 64 W
  const int s_total = M * KB;
  float sv[2] = {0.f, 0.f}, wsv = 0.f;                       // (M * K / 128 <= 1024)
  if (MODE == QD_BLOCK) {
#pragma unroll
    for (int p = 0; p < 2; ++p) sv[p] = a.x_scale[min(tid + p * THREADS, s_total - 1)];
    wsv = a.w_scale[(n0 >> 7) * KB + min(tid, KB - 1)];
  }
  __builtin_amdgcn_sched_barrier(0);

  const rsrc_t wres = make_rsrc(a.w, (uint32_t)N * (uint32_t)K);
  const uint32_t kstride = a.kslab ? 8192 : 128, vstride = a.kslab ? 1024 : 16;
  uint32_t woff[NI];
#pragma unroll
  for (int t = 0; t < NI; ++t) {
    const int n = n0 + 16 * t;
    woff[t] = n >= N ? FEW_NONE : a.kslab ? few_kslab_offset(n, KB, lane) : (uint32_t)((n + r16) * K + 32 * q);
  }
  FewWeights<NI, BPR> ring;
  auto ask = [&](int b, int kb) { ring.ask(b, wres, woff, kb, KB, kstride, vstride); };
#pragma unroll
  for (int b = 0; b < BPR; ++b) ask(b, wave + W * b);
  __builtin_amdgcn_sched_barrier(0);

  // ---- x into LDS as codes
  if (SRC == QD_TOKEN) {
    few_lds_barrier();                                        // row_max is cleared
#pragma unroll
    for (int p = 0; p < PIECES; ++p) {
      if (p * THREADS >= total) break;
      const int i = tid + p * THREADS;
      float y[8], mx = 0.f;
      unpack8<DT>(xv[p], y);
#pragma unroll
      for (int e = 0; e < 8; ++e) mx = fmaxf(mx, fabsf(y[e]));
      mx = lane_group_max(mx, 16);                           // (a row is a whole number of sixteen pieces)
      if ((lane & 15) == 0 && i < total) atomicMax(&row_max[a.row_pieces.div((uint32_t)i)], bitcast<uint32_t>(mx));
    }
    few_lds_barrier();
  }
#pragma unroll
  for (int p = 0; p < PIECES; ++p) {
    if (p * THREADS >= total) break;
    const int i = tid + p * THREADS;
    const int r = (int)a.row_pieces.div((uint32_t)min(i, total - 1)), c = i - r * (int)a.row_pieces.d;
    if (SRC == QD_CODES) {
      if (i < total) *(u4*)(lds + few_chunk_at(M, c >> 3, r, c & 7)) = xv[p];
    } else {
      float y[8];
      unpack8<DT>(xv[p], y);
      u2 codes;
      if constexpr (SRC == QD_CHANNEL) {
        float s[8];
        unpack8<DT>(cv[p], s);
        codes = static_int8_codes<DT>(y, s);
      } else if constexpr (MODE == QD_INT8) {
        codes = RowInt8(bitcast<float>(row_max[r])).codes(y);
      } else {
        codes = RowFp8(bitcast<float>(row_max[r])).codes(y);
      }
      if (i < total) *(u2*)(lds + few_chunk_at(M, c >> 4, r, (c & 15) >> 1) + (c & 1) * 8) = codes;
    }
  }
  float* const xs_l = (float*)(lds + (size_t)M * K);         // [row][K block], then the columns' scales
  float* const ws_l = xs_l + s_total;
  if (MODE == QD_BLOCK) {
#pragma unroll
    for (int p = 0; p < 2; ++p)
      if (tid + p * THREADS < s_total) xs_l[tid + p * THREADS] = sv[p];
    if (tid < KB) ws_l[tid] = wsv;
  }
  static_assert(SRC != QD_TOKEN || MT == 1, "sixteen largest magnitudes");
  if (SRC == QD_TOKEN && stores)
    xs[0] = MODE == QD_INT8 ? RowInt8(bitcast<float>(row_max[r16])).scale : RowFp8(bitcast<float>(row_max[r16])).scale;
  few_lds_barrier();

  // ---- K blocks wave, wave + W, ..
  acc_t acc[MT][NI];
#pragma unroll
  for (int j = 0; j < MT; ++j)
#pragma unroll
    for (int t = 0; t < NI; ++t) acc[j][t] = (acc_t){0, 0, 0, 0};
  int row[MT];
#pragma unroll
  for (int j = 0; j < MT; ++j) row[j] = min(16 * j + r16, M - 1);
  auto multiply = [&](int b, int kb) {
#pragma unroll
    for (int j = 0; j < MT; ++j) {
      const FewOperand x(lds, M, kb, row[j], q);
      const float sc = MODE == QD_BLOCK ? xs_l[row[j] * KB + kb] * ws_l[kb] : 1.0f;
#pragma unroll
      for (int t = 0; t < NI; ++t) {
        if constexpr (MODE == QD_INT8) {
#pragma unroll
          for (int v = 0; v < 2; ++v) acc[j][t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(bitcast<i4>(ring.w[b][t][v]), bitcast<i4>(x.v[v]), acc[j][t], 0, 0, 0);
        } else if constexpr (MODE == QD_BLOCK) {
          acc[j][t] += sc * few_fp8_products(ring.w[b][t], x, (f4){0.f, 0.f, 0.f, 0.f});
        } else {
          acc[j][t] = few_fp8_products(ring.w[b][t], x, acc[j][t]);
        }
      }
    }
  };
  few_walk<BPR, W>(KB, wave, multiply, ask);

  // ---- the wavefronts' sums, in wavefront order
  few_lds_barrier();                                          // everybody has read x
  acc_t* const red = (acc_t*)lds;
#pragma unroll
  for (int j = 0; j < MT; ++j)
#pragma unroll
    for (int t = 0; t < NI; ++t) red[(wave * NI * MT + j * NI + t) * 64 + lane] = acc[j][t];
  few_lds_barrier();
  if (!stores) return;
#pragma unroll
  for (int f = 0; f < FIN; ++f) {
    const int m = stored_row(f);
    if (m >= M) return;
    const acc_t sum = few_sum<W>(red, NI * MT, wave + W * f, lane);
    float v[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      v[e] = MODE == QD_BLOCK ? (float)sum[e] : scaled_sum((float)sum[e], xs[f], ws[e]);
      const uint32_t bw = e < 2 ? bs.x : bs.y;
      if (a.bias) v[e] = plus_bias(v[e], Elem<DT>::to_f32((uint16_t)((e & 1) ? bw >> 16 : bw & 0xffffu)));
    }
    u2 o;
    o.x = (uint32_t)Elem<DT>::from_f32(v[0]) | ((uint32_t)Elem<DT>::from_f32(v[1]) << 16);
    o.y = (uint32_t)Elem<DT>::from_f32(v[2]) | ((uint32_t)Elem<DT>::from_f32(v[3]) << 16);
    *(u2*)((uint16_t*)a.out + (size_t)m * N + nt) = o;
  }
}

// column tiles per workgroup: one workgroup per CU
int qd_tiles(int N) {
  const int cus = device_cu_count();
  for (int ni = 1; ni <= 8; ni *= 2)
    if ((N + 16 * ni - 1) / (16 * ni) <= cus) return ni;
  return 0;
}
size_t qd_lds_bytes(int mode, int M, int K, int ni, int waves) {
  const size_t x = (size_t)M * K + (mode == QD_BLOCK ? ((size_t)M * (K / 128) + K / 128) * 4 : 0), sums = (size_t)waves * ni * ((M + 15) / 16) * 1024;
  return x > sums ? x : sums;
}
// (with four wavefronts K blocks are added in the order of kcontig_gemm_kernel, which takes codes of so short a K)
int qd_waves(int K) { return K < 2048 ? 4 : 8; }

// What q8_decode_tiles and quant_tiles can ask for, and is built.  Codes of up to 16 rows and rows for eight wavefronts have two K blocks to a wavefront at least, rows for
// four (K below 2048) four at most; taller rows are as deep as their KiB allow; and the large layers of 17 .. 32 rows have four or eight column tiles and four K
// blocks to a wavefront at least.
constexpr bool qd_built(int mode, int src, int ni, int waves, int bpr, int mt) {
  if (src != QD_CODES) return mt == 1 && (waves == 4 ? ni < 8 && bpr <= 4 : ni == 8 || bpr > 1);
  if (mt == 1 || ni == 8) return mt <= 2 && (ni == 8 || bpr > 1);
  if (mt == 2) return ni == 1 || (ni == 2 ? mode == QD_BLOCK || (mode == QD_INT8 && bpr <= 2) : mode == QD_INT8 || bpr == 2);
  if (mt == 3) return bpr <= 4 && (mode == QD_INT8 || (mode == QD_BLOCK && ni <= 2));
  return mode == QD_INT8 && ni >= 2 && bpr <= 2;
}

template <int MODE, int SRC, int DT, int NI, int W, int BPR, int MT>
int launch_qd_rows(const QdArgs& a, hipStream_t st) {
  if constexpr (qd_built(MODE, SRC, NI, W, BPR, MT)) {
    static hipError_t attr = hipFuncSetAttribute((const void*)q8_decode_kernel<MODE, SRC, DT, NI, W, BPR, MT>, hipFuncAttributeMaxDynamicSharedMemorySize, 144 * 1024);
    MQ_REQUIRE(attr == hipSuccess, "q8_decode: cannot reserve LDS: %s", hipGetErrorString(attr));
    hipLaunchKernelGGL((q8_decode_kernel<MODE, SRC, DT, NI, W, BPR, MT>), dim3((a.N + 16 * NI - 1) / (16 * NI)), dim3(64 * W), qd_lds_bytes(MODE, a.M, a.K, NI, W), st, a);
    MQ_LAUNCH_CHECK("q8_decode");
    return 0;
  }
  MQ_REQUIRE(false, "q8_decode: M=%d N=%d K=%d is not covered", a.M, a.N, a.K);
}
template <int MODE, int SRC, int DT, int NI, int W, int BPR>
int launch_qd(const QdArgs& a, hipStream_t st) {
  switch ((a.M + 15) / 16) {
    case 1: return launch_qd_rows<MODE, SRC, DT, NI, W, BPR, 1>(a, st);
    case 2: return launch_qd_rows<MODE, SRC, DT, NI, W, BPR, 2>(a, st);
    case 3: return launch_qd_rows<MODE, SRC, DT, NI, W, BPR, 3>(a, st);
    default: return launch_qd_rows<MODE, SRC, DT, NI, W, BPR, 4>(a, st);
  }
}
template <int MODE, int SRC, int DT, int NI, int W>
int launch_qd_ring(const QdArgs& a, hipStream_t st) {
  const int blocks = (a.K / 128 + W - 1) / W;        // of a wavefront: what lies beyond the last costs its requests
  if constexpr (NI <= 1) if (blocks > 4) return launch_qd<MODE, SRC, DT, NI, W, 8>(a, st);
  if constexpr (NI <= 2) if (blocks > 2) return launch_qd<MODE, SRC, DT, NI, W, 4>(a, st);
  if constexpr (NI <= 4) if (blocks > 1) return launch_qd<MODE, SRC, DT, NI, W, 2>(a, st);
  return launch_qd<MODE, SRC, DT, NI, W, 1>(a, st);
}
template <int MODE, int SRC, int DT, int W>
int launch_qd_tiles(const QdArgs& a, int tiles, hipStream_t st) {
  switch (tiles) {
    case 1: return launch_qd_ring<MODE, SRC, DT, 1, W>(a, st);
    case 2: return launch_qd_ring<MODE, SRC, DT, 2, W>(a, st);
    case 4: return launch_qd_ring<MODE, SRC, DT, 4, W>(a, st);
    default: return launch_qd_ring<MODE, SRC, DT, 8, W>(a, st);
  }
}
template <int MODE, int SRC, int DT>
int launch_qd_waves(const QdArgs& a, int tiles, hipStream_t st) {
  if constexpr (SRC != QD_CODES) if (qd_waves(a.K) == 4) return launch_qd_tiles<MODE, SRC, DT, 4>(a, tiles, st);
  return launch_qd_tiles<MODE, SRC, DT, 8>(a, tiles, st);
}

}  // namespace

// Column tiles per workgroup where codes of M rows go here, 0 where they do not.  The rows fill LDS at 128 KiB.
//  - Up to 16 rows, against kcontig_gemm_kernel, 1700 launches with weights from memory and from the cache: below K 2048 that is ahead (1024 x 4096 at one row
//    3.0 us against 3.5), and with two column tiles per workgroup its wavefronts catch up from 96 KiB on (8192 x 8192 at 16 rows 12.2 us against 12.9).  Block scales: from 6144
//    columns on it has 32 columns to a workgroup as well, and is up to 9 % ahead over K 2560 .. 16384 (one row), and 64 from 12288 (up to 5 %, to four rows).
//    Row-major weights, a tile of which is sixteen pieces K bytes apart: with two or four column tiles and a long K that is ahead (there / here, one row: block scales
//    16384 x 8192 0.75, 12288 x 8192 0.88, 4096 x 14336 0.89, 8192 x 16384 0.80; scales outside 8192 x 16384 0.89, 12288 x 14336 0.92), with one and eight column tiles
//    at no K (1.04 and more).
//  - 17 .. 64 rows, against q8_mid_kernel, which reads a share of the rows for every 32 or 64 columns and walks K through a barrier per block: 22 layers of K 1024 .. 7168 at nine
//    numbers of rows, with weights from memory and from the last-level cache.  From memory this is ahead nearly everywhere (1.0 .. 1.7 times); from the cache the copy of all rows into every
//    workgroup costs more than the weights, so the lines are where that pays less than 4 %.  (us, from memory, there / here, and the ratio from the cache: block scales 2048 x 2048 at 20 6.0 /
//    3.5, 1.68, 2048 x 7168 at 24 / 48 6.2 / 5.3, 1.23, 6.9 / 6.5, 1.02, 4096 x 12288 at 24 13.2 / 12.6, 0.95; int8 4096 x 4096 at 24 7.8 / 6.0, 1.10, 3584 x 4608 at 20 7.2 / 6.2, 1.00, 4096 x 6144 at 24
//    8.3 / 7.3, 0.91, 2048 x 11008 at 24 / 48 8.3 / 6.9, 1.09, 10.4 / 7.9, 1.07; per channel 4096 x 4096 at 20 / 32 7.9 / 5.9, 1.39, 8.0 / 7.0, 0.97, 3072 x 4608 at 24 6.6 / 6.3, 0.92;
//    block scales at 40 rows 3200 x 8192 0.92, from the cache 0.90, 3200 x 5120 1.00, 1.00; int8 at 24 3584 x 8320 1.15, 0.91, at 28 3072 x 11264 1.12, 1.00.)
//  - 17 .. 32 rows of large layers, against the streamer (5120 x 13824 at 24, int8 16.2 / 15.0 and 1.08; 4096 x 28672 at 32 25.1 / 22.6 and 1.11).
int q8_decode_tiles(int mode, int M, int N, int K, bool kslab) {
  if (M < 1 || M > 64 || K % 128 != 0 || K > 65536 || N % 16 != 0 || (long)M * K > 128 * 1024 || (size_t)N * K >= ((size_t)1 << 31)) return 0;
  const int tiles = qd_tiles(N), rows = (M + 15) / 16;
  if (M <= 16) {
    bool no = K < 2048 || (tiles == 2 && M * K > 96 * 1024);
    if (kslab) no |= mode == QD_BLOCK && ((tiles == 2 && N >= 6144 && (K > 2048 || M <= 4)) || (tiles == 4 && N >= 12288 && M <= 4));
    else if (tiles == 2) no |= mode == QD_BLOCK && K > 6144 && M <= 4;
    else if (tiles == 4) no |= mode == QD_BLOCK ? K >= 4096 && (M <= 8 || N > 12544) : K >= 8192 && N > 12544;
    return no ? 0 : tiles;
  }
  if (!kslab || K < 1024) return 0;
  if (M <= 32 && N >= 12288 && (long)K * N >= (1L << 26)) return tiles;
  if (tiles > 4) return 0;
  int most = 0;                                              // KiB of rows
  if (mode == QD_BLOCK) {
    if (rows == 2) most = tiles == 1 ? 128 : tiles == 2 ? 100 : 0;
    else if (rows == 3 && tiles <= 2) most = K <= 2048 || (M <= 40 && N <= 5120) ? 128 : 0;
  } else if (mode == QD_PC) {
    most = tiles == 1 && rows == 2 ? 96 : 0;
  } else if (rows == 2) {
    most = tiles == 1 ? 112 : tiles == 2 ? (K <= 2048 ? 64 : 0) : K <= 2048 || N >= 11008 ? 96 : 0;
  } else if (rows == 3) {
    most = tiles == 1 ? (M <= 40 ? 96 : 0) : tiles == 2 ? 120 : 112;
  } else {
    most = tiles >= 2 ? 64 : 0;
  }
  return M * K <= most * 1024 ? tiles : 0;
}

// (the loads and stores of its widths)
bool q8_decode_reads(const void* x, const void* w, const void* w_scale, const void* bias, const void* out) {
  return (((size_t)x | (size_t)w | (size_t)w_scale) & 15) == 0 && (((size_t)bias | (size_t)out) & 7) == 0;
}

// Whether 16-bit rows are quantised here.  Every workgroup quantises all of them, 0.12 us per 1024 elements, which is ahead of a launch that does it once up
// to some 16000 (4096 x 4096 at 4 rows, fp8: 8.0 -> 6.5 us; 2048 x 7168 at 8 7.0 -> 6.4; 1024 x 4096 at 16 5.8 -> 5.3); one long row takes that launch longer than
// several short ones.
static int quant_tiles(int mode, int quant, int M, int N, int K) {
  if (M < 1 || M > 16 || K % 128 != 0 || N % 64 != 0 || (long)M * K > (M == 1 ? 20480 : 16384) || (size_t)N * K >= ((size_t)1 << 31)) return 0;
  if (mode == QD_PC ? quant != QD_TOKEN : mode != QD_INT8 || (quant != QD_TOKEN && quant != QD_CHANNEL)) return 0;
  const int tiles = qd_tiles(N);
  return tiles <= qd_waves(K) ? tiles : 0;
}

int q8_decode_launch(int tiles, int mode, int src, void* out, const void* x, const void* w, const float* x_scale, int sc_row, const void* c_scale,
                     const float* w_scale, int sc_col, const void* bias, int M, int N, int K, int kslab, int dtype, hipStream_t st) {
  MQ_REQUIRE(dtype == MI355Q_F16 || dtype == MI355Q_BF16, "q8_decode: output dtype %d must be f16 or bf16", dtype);
  QdArgs a = {};
  a.out = out; a.x = x; a.w = (const uint8_t*)w; a.x_scale = x_scale; a.c_scale = (const uint16_t*)c_scale; a.w_scale = w_scale;
  a.bias = (const uint16_t*)bias;
  a.sc_row = sc_row; a.sc_col = sc_col;
  a.M = M; a.N = N; a.K = K; a.kslab = kslab;
  a.row_pieces = FastDiv((uint32_t)(K / (src == QD_CODES ? 16 : 8)));
#define QD_CASE(MODE_, SRC_) \
  if (mode == MODE_ && src == SRC_) return dtype == MI355Q_F16 ? launch_qd_waves<MODE_, SRC_, MI355Q_F16>(a, tiles, st) : launch_qd_waves<MODE_, SRC_, MI355Q_BF16>(a, tiles, st)
  QD_CASE(QD_BLOCK, QD_CODES);
  QD_CASE(QD_PC, QD_CODES);
  QD_CASE(QD_PC, QD_TOKEN);
  QD_CASE(QD_INT8, QD_CODES);
  QD_CASE(QD_INT8, QD_TOKEN);
  QD_CASE(QD_INT8, QD_CHANNEL);
#undef QD_CASE
  MQ_REQUIRE(false, "q8_decode: mode %d with rows of kind %d", mode, src);
}

}  // namespace mi355q

using namespace mi355q;

extern "C" int mi355q_q8_quant_gemm_takes(int kind, int quant, int M, int N, int K) { return quant_tiles(kind, quant, M, N, K) > 0; }

extern "C" int mi355q_q8_quant_gemm(void* out, const void* x, const void* w, const void* x_scale, const float* w_scale, int w_scale_per_col,
                                    const void* bias, int kind, int quant, int M, int N, int K, int dtype, void* stream) {
  MQ_REQUIRE(M >= 0 && N > 0 && K > 0, "q8_quant_gemm: bad shape M=%d N=%d K=%d", M, N, K);
  if (M == 0) return 0;
  MQ_REQUIRE(dtype == MI355Q_F16 || dtype == MI355Q_BF16, "q8_quant_gemm: dtype %d must be f16 or bf16", dtype);
  const int tiles = quant_tiles(kind, quant, M, N, K);
  MQ_REQUIRE(tiles > 0, "q8_quant_gemm: kind %d, quantiser %d, M=%d N=%d K=%d is not covered (mi355q_q8_quant_gemm_takes)", kind, quant, M, N, K);
  MQ_REQUIRE(out && x && w && w_scale && (quant != QD_CHANNEL || x_scale), "q8_quant_gemm: null pointer");
  MQ_REQUIRE((((size_t)x | (size_t)w | (quant == QD_CHANNEL ? (size_t)x_scale : 0) | (w_scale_per_col ? (size_t)w_scale : 0)) & 15) == 0 &&
             (((size_t)out | (size_t)bias) & 7) == 0, "q8_quant_gemm: x, the weights and the scales must be aligned to 16 bytes, out and bias to 8");
  return q8_decode_launch(tiles, kind, quant, out, x, w, nullptr, 0, x_scale, w_scale, w_scale_per_col ? 1 : 0, bias, M, N, K, 1, dtype, as_stream(stream));
}
