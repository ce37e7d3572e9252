// fp8 experts (128 x 128 block scales) on up to 64 slots of up to four tokens, where the experts that they reach are too few to fill the chip with
// workgroups of 256 columns.
//
// The sorted launches give an expert 2 I / 256 workgroups and then K / 256, each with four wavefronts: a token of eight experts of 2048 x 4608 and 2304 x 1152 has
// 72 of them on 256 CUs, and its weights arrive at 2 TB/s.  Here a workgroup has 16 .. 128 columns and eight wavefronts that share K, each with up to
// eight tiles x one K block on their way (as q8_decode_kernel, whose measurements of that hold); it finds its block of slots in the ids by itself and
// quantises the block's rows -- the tokens' rows for the first GEMM, gate and up with the activation for the second -- while the weights arrive, so that the
// alignment and both quantisers are no launches.  Bound by the memory system: workgroups per CU come out uneven, and the rows of a block are quantised by every
// workgroup of the expert (0.12 .. 0.3 us per 1024 values).
//
// Measured (us in a graph, alignment to sum, weights out of the caches, the sorted launches -> here): eight experts to a token, 128 of 2304 / 1152 at 1 / 2 / 3 tokens 35.9 / 38.2 / 44.1
// -> 25.8 / 35.5 / 42.5; 128 of 4096 / 1024 45.0 / 49.1 / 61.6 -> 26.6 / 41.5 / 57.8; 256 of 7168 / 2048 at 1 74.8 -> 64.2; six to a token, 128 of 6144 / 512 at 1 / 2 / 3
// 48.3 / 53.9 / 56.8 -> 23.2 / 37.2 / 48.1.
#include "moe_slots.h"
#include "q8_few.h"

#include <algorithm>
#include <cmath>

namespace mi355q {

int moe_sum_launch(void* out, const void* in, long rows, int topk, int K, int in_dtype, int out_dtype, const int32_t* valid_rows, const int32_t* ids,
                   int id_step, int E, hipStream_t st);

namespace {

struct QeArgs {
  uint16_t* out;                // [numel, N]
  const uint16_t* x;            // rows [tokens, K], or gate and up columns [numel, 2 K]
  const uint8_t* w;             // [E, N, K], kslab order
  const float* w_scale;         // [E, N / 128, K / 128]
  const float* topk_weights;    // [numel] or null
  const int32_t* ids;           // the slots' experts, every id_step'th int32
  int id_step, id_bits, numel, topk, E;
  int N, K;
  FastDiv row_pieces;           // pieces of 8 values in a row
};

constexpr int QE_W = 8, QE_PIECES = 4, SHIFT = 2;            // (a token has an expert once: a block of four slots takes all rows that four tokens give it)

// GATED: x holds gate and up, and what is quantised is what silu_and_mul makes of them; else the rows of the slots' tokens.  NI tiles of 16 columns,
// eight wavefronts that take the K blocks in turn, BPR K blocks of each on their way; blocks of 2^SHIFT slots.
template <bool GATED, int DT, int NI, int BPR>
__global__ void __launch_bounds__(64 * QE_W, 2)
q8_experts_kernel(QeArgs a) {
  constexpr int THREADS = 64 * QE_W, XL = GATED ? 2 : 1;
  extern __shared__ __align__(16) unsigned char lds[];       // x: [K block][row][eight chunks of 16 bytes], scales; then the wavefronts' sums
  __shared__ int slot_of[16];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15, q = lane >> 4;
  const int N = a.N, K = a.K, KB = K >> 7;
  const SlotBlock blk = find_slot_block<SHIFT>(a.ids, a.id_step, a.id_bits, a.numel, a.E, (int)blockIdx.y, lane);
  if (!blk.real) return;
  const int R = blk.real;
  if (wave == 0 && holds_lane<SHIFT>(blk)) slot_of[blk.rank & ((1 << SHIFT) - 1)] = lane;
  __syncthreads();
  const int n0 = xcd_tile() * (16 * NI);

  // ---- requests: rows first, then weights
  const int total = R * (int)a.row_pieces.d;
  u4 xv[QE_PIECES][XL];
  auto ask_x = [&](int p, int first) {
    const int i = min(first + tid + p * THREADS, total - 1);
    const int r = (int)a.row_pieces.div((uint32_t)i), c = i - r * (int)a.row_pieces.d, slot = slot_of[r];
    const uint16_t* row = a.x + (GATED ? (size_t)slot * 2 * K : (size_t)(slot / a.topk) * K) + 8 * c;
    xv[p][0] = *(const u4*)row;
    if constexpr (GATED) xv[p][1] = *(const u4*)(row + K);
  };
#pragma unroll
  for (int p = 0; p < QE_PIECES; ++p) {
    if (p * THREADS >= total) break;
    ask_x(p, 0);
  }
  const int nt = n0 + 16 * wave + 4 * q;                     // columns of the outputs that this lane stores (wave < NI)
  const bool stores = wave < NI && nt < N;
  const float* const wsc = a.w_scale + ((size_t)blk.expert * ((N + 127) >> 7) + (n0 >> 7)) * KB;
  const float wsv = wsc[min(tid, KB - 1)];
  __builtin_amdgcn_sched_barrier(0);
  const rsrc_t wres = make_rsrc(a.w + (size_t)blk.expert * N * K, (uint32_t)N * (uint32_t)K);
  uint32_t woff[NI];
#pragma unroll
  for (int t = 0; t < NI; ++t) woff[t] = n0 + 16 * t >= N ? FEW_NONE : few_kslab_offset(n0 + 16 * t, KB, lane);
  FewWeights<NI, BPR> ring;
  auto ask = [&](int b, int kb) { ring.ask(b, wres, woff, kb, KB, 8192, 1024); };
#pragma unroll
  for (int b = 0; b < BPR; ++b) ask(b, wave + QE_W * b);
  __builtin_amdgcn_sched_barrier(0);

  // ---- rows into LDS as codes with a scale per 128 values (sixteen lanes)
  float* const xs_l = (float*)(lds + (size_t)R * K);         // [row][K block], then the columns' scales
  float* const ws_l = xs_l + R * KB;
  auto quantise = [&](int p, int first) {
    const int i = first + tid + p * THREADS, at = min(i, total - 1);
    const int r = (int)a.row_pieces.div((uint32_t)at), c = at - r * (int)a.row_pieces.d;
    float y[8], mx = 0.f;
    unpack8<DT>(xv[p][0], y);
    if constexpr (GATED) {
      float up[8];
      unpack8<DT>(xv[p][1], up);
#pragma unroll
      for (int e = 0; e < 8; ++e) y[e] = round_act<DT>(silu_mul(y[e], up[e]));
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) mx = fmaxf(mx, fabsf(y[e]));
    const RowFp8 by(lane_group_max(mx, 16));                 // (a row is a whole number of sixteen pieces)
    const u2 codes = by.codes(y);
    if (i < total) {
      *(u2*)(lds + few_chunk_at(R, c >> 4, r, (c & 15) >> 1) + (c & 1) * 8) = codes;
      if ((c & 15) == 0) xs_l[r * KB + (c >> 4)] = by.scale;
    }
  };
#pragma unroll
  for (int p = 0; p < QE_PIECES; ++p) {
    if (p * THREADS >= total) break;
    quantise(p, 0);
  }
  for (int first = QE_PIECES * THREADS; first < total; first += THREADS) {   // (many rows: a piece at a time, behind the weights)
    ask_x(0, first);
    quantise(0, first);
  }
  for (int i = tid; i < KB; i += THREADS) ws_l[i] = i == tid ? wsv : wsc[i];
  few_lds_barrier();

  // ---- K blocks wave, wave + 8, ..
  f4 acc[NI];
#pragma unroll
  for (int t = 0; t < NI; ++t) acc[t] = (f4){0.f, 0.f, 0.f, 0.f};
  const int row = min(r16, R - 1);
  auto multiply = [&](int b, int kb) {
    const FewOperand x(lds, R, kb, row, q);
    const float sc = xs_l[row * KB + kb] * ws_l[kb];
#pragma unroll
    for (int t = 0; t < NI; ++t) acc[t] += sc * few_fp8_products(ring.w[b][t], x, (f4){0.f, 0.f, 0.f, 0.f});
  };
  few_walk<BPR, QE_W>(KB, wave, multiply, ask);

  // ---- the wavefronts' sums, in wavefront order
  few_lds_barrier();                                          // everybody has read x
  f4* const red = (f4*)lds;
#pragma unroll
  for (int t = 0; t < NI; ++t) red[(wave * NI + t) * 64 + lane] = acc[t];
  few_lds_barrier();
  if (!stores || r16 >= R) return;
  const f4 sum = few_sum<QE_W>(red, NI, wave, lane);
  const int slot = slot_of[r16];
  const float rw = a.topk_weights ? a.topk_weights[slot] : 1.0f;
  u2 o;
  o.x = (uint32_t)Elem<DT>::from_f32(sum[0] * rw) | ((uint32_t)Elem<DT>::from_f32(sum[1] * rw) << 16);
  o.y = (uint32_t)Elem<DT>::from_f32(sum[2] * rw) | ((uint32_t)Elem<DT>::from_f32(sum[3] * rw) << 16);
  *(u2*)(a.out + (size_t)slot * N + nt) = o;
}

size_t qe_lds_bytes(int rows, int K, int ni) {
  const int KB = K / 128;
  return std::max((size_t)rows * K + (size_t)(rows + 1) * KB * 4, (size_t)QE_W * ni * 1024);
}
// experts that evenly spread slots reach
double qe_hit(int numel, int E) { return E * (1.0 - std::pow(1.0 - 1.0 / E, numel)); }
// A workgroup's column tiles: the fewest with which there are some three workgroups per CU at most (as many as CUs: one token of six of 64 experts of 7168 / 2048
// 56.5 us against 51.4, two tokens of eight of 128 of 2304 / 1152 41.0 against 35.5; nowhere ahead by more than 2 us)
int qe_tiles(int numel, int E, int N) {
  const double hit = qe_hit(numel, E);
  int ni = 1;
  while (ni < 8 && hit * N / (16 * ni) > 3.2 * device_cu_count()) ni *= 2;
  return ni;
}

template <bool GATED, int DT, int NI, int BPR>
int launch_qe(const QeArgs& a, hipStream_t st) {
  static hipError_t attr = hipFuncSetAttribute((const void*)q8_experts_kernel<GATED, DT, NI, BPR>, hipFuncAttributeMaxDynamicSharedMemorySize, 144 * 1024);
  MQ_REQUIRE(attr == hipSuccess, "moe_fp8_unsorted: cannot reserve LDS: %s", hipGetErrorString(attr));
  const int blocks = std::min(a.numel, a.E + (a.numel >> SHIFT));
  hipLaunchKernelGGL((q8_experts_kernel<GATED, DT, NI, BPR>), dim3((a.N + 16 * NI - 1) / (16 * NI), blocks), dim3(64 * QE_W),
                     qe_lds_bytes(std::min(a.numel, 1 << SHIFT), a.K, NI), st, a);
  MQ_LAUNCH_CHECK("moe_fp8_unsorted");
  return 0;
}
template <bool GATED, int DT, int NI>
int launch_qe_ring(const QeArgs& a, hipStream_t st) {
  const int blocks = (a.K / 128 + QE_W - 1) / QE_W;  // of a wavefront
  if constexpr (NI <= 1) if (blocks > 4) return launch_qe<GATED, DT, NI, 8>(a, st);
  if constexpr (NI <= 2) if (blocks > 2) return launch_qe<GATED, DT, NI, 4>(a, st);
  if constexpr (NI <= 4) if (blocks > 1) return launch_qe<GATED, DT, NI, 2>(a, st);
  return launch_qe<GATED, DT, NI, 1>(a, st);
}
template <bool GATED, int DT>
int launch_qe_tiles(const QeArgs& a, hipStream_t st) {
  switch (qe_tiles(a.numel, a.E, a.N)) {
    case 1: return launch_qe_ring<GATED, DT, 1>(a, st);
    case 2: return launch_qe_ring<GATED, DT, 2>(a, st);
    case 4: return launch_qe_ring<GATED, DT, 4>(a, st);
    default: return launch_qe_ring<GATED, DT, 8>(a, st);
  }
}
}  // namespace
}  // namespace mi355q

using namespace mi355q;

extern "C" size_t mi355q_moe_fp8_unsorted_bytes(int M, int topk, int E, int K, int I) {
  if (M < 1 || topk < 1 || E < 1 || K < 128 || I < 128 || K % 128 || I % 128 || M > 64 / topk || M > 4) return 0;
  const int numel = M * topk, rows = std::min(numel, 1 << SHIFT);
  if ((size_t)2 * I * K >= ((size_t)1 << 31) || (size_t)rows * std::max(K, I) > 128 * 1024) return 0;
  return (size_t)numel * (2 * I + K) * 2;
}

// The line: while the sorted launches would have fewer than two workgroups of 256 columns per CU in both GEMMs together.  There this is ahead by 4 .. 100 %
// (seven pairs of K and I); beyond, and at five to eight tokens, it is 10 % ahead to 17 % behind.
extern "C" int mi355q_moe_fp8_unsorted_wanted(int M, int topk, int E, int K, int I) {
  return mi355q_moe_fp8_unsorted_bytes(M, topk, E, K, I) > 0 && qe_hit(M * topk, E) * (2.0 * I + K) < 2.0 * 256 * device_cu_count();
}

extern "C" int mi355q_moe_fp8_unsorted(void* out, const void* x, const void* w1, const float* w1_scale, const void* w2, const float* w2_scale,
                                       const float* topk_weights, const void* topk_ids, int ids_are_int64, int M, int topk, int E, int K, int I, int dtype,
                                       void* workspace, size_t workspace_bytes, void* stream) {
  MQ_REQUIRE(M >= 0 && topk > 0 && E > 0 && K > 0 && I > 0, "moe_fp8_unsorted: bad shape");
  if (M == 0) return 0;
  const size_t need = mi355q_moe_fp8_unsorted_bytes(M, topk, E, K, I);
  MQ_REQUIRE(need > 0, "moe_fp8_unsorted: M=%d topk=%d E=%d K=%d I=%d is not covered", M, topk, E, K, I);
  MQ_REQUIRE(out && x && w1 && w1_scale && w2 && w2_scale && topk_weights && topk_ids && workspace && workspace_bytes >= need, "moe_fp8_unsorted: null pointer, or a workspace below %zu bytes", need);
  MQ_REQUIRE((((size_t)out | (size_t)x | (size_t)w1 | (size_t)w2 | (size_t)workspace) & 15) == 0, "moe_fp8_unsorted: operands must be aligned to 16 bytes");
  MQ_REQUIRE(dtype == MI355Q_F16 || dtype == MI355Q_BF16, "moe_fp8_unsorted: dtype %d", dtype);
  hipStream_t st = as_stream(stream);
  uint16_t* const down = (uint16_t*)workspace;
  uint16_t* const gate_up = down + (size_t)M * topk * K;
  QeArgs a = {};
  a.ids = (const int32_t*)topk_ids; a.id_step = ids_are_int64 ? 2 : 1;
  while ((1 << a.id_bits) < E) ++a.id_bits;
  a.numel = M * topk; a.E = E;
  a.out = gate_up; a.x = (const uint16_t*)x; a.w = (const uint8_t*)w1; a.w_scale = w1_scale; a.topk = topk; a.N = 2 * I; a.K = K; a.row_pieces = FastDiv(K / 8);
  int rc = dtype == MI355Q_F16 ? launch_qe_tiles<false, MI355Q_F16>(a, st) : launch_qe_tiles<false, MI355Q_BF16>(a, st);
  if (rc) return rc;
  a.out = down; a.x = gate_up; a.w = (const uint8_t*)w2; a.w_scale = w2_scale; a.topk_weights = topk_weights; a.topk = 1; a.N = K; a.K = I; a.row_pieces = FastDiv(I / 8);
  rc = dtype == MI355Q_F16 ? launch_qe_tiles<true, MI355Q_F16>(a, st) : launch_qe_tiles<true, MI355Q_BF16>(a, st);
  if (rc) return rc;
  return moe_sum_launch(out, down, M, topk, K, dtype, dtype, nullptr, a.ids, a.id_step, E, st);
}
