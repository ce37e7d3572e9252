// Elementwise glue between the GEMMs: SiLU-gate, fp8-e4m3fn activation
// quantisers (per token group, per token, static), the fused SiLU-gate + group
// quantiser, and the top-k sum: 16-byte loads per lane,
// fp32 arithmetic, one pass over the data.  The sum, the plain gate and the per-token quantisers are HBM-bound; norm and gate with group codes were bound by
// their instructions (33 and 61 per element), of which conversions in pairs, a maximum and a division of three instructions each and a reciprocal of
// as many are left (us, bf16, rows 1537 / 4096 x 7168: norm + codes 11.5 / 24.4 -> 9.9 / 20.4, gate + codes 15.9 / 36.5 -> 11.7 / 28.1, codes alone
// 7.0 / 16.1 -> 6.2 / 14.9).  Every kernel takes an optional
// device int32 `valid_rows` so padded (graph-captured) batches skip dead rows
// without a host synchronisation.
#include "moe_align.h"
#include "rows8.h"

#include <algorithm>

namespace mi355q {
namespace {


template <int DT> struct E16 { typedef Elem<DT> T; };

template <int DT>
__device__ __forceinline__ u4 pack8(const float* f) {
  u4 v;
#pragma unroll
  for (int i = 0; i < 4; ++i)
    v[i] = (uint32_t)Elem<DT>::from_f32(f[2 * i]) | ((uint32_t)Elem<DT>::from_f32(f[2 * i + 1]) << 16);
  return v;
}
// Rows of this launch that count: `rows` of them, or up to the device's row count (times rows per count) less the `row0` rows of
// the launches before this one.
__device__ __forceinline__ uint32_t live_rows(uint32_t rows, const int* valid_rows, int rpc, long row0) {
  return valid_rows ? (uint32_t)max(0L, min((long)rows, (long)max(0, *valid_rows) * rpc - row0)) : rows;
}

// ---- silu_and_mul: out[r, :d] = silu(x[r, :d]) * x[r, d:] -------------------
// (row and piece of an item by multiplication: a 64-bit division per 16-byte piece was a quarter of these kernels'
// instructions, and they are bound by issue as much as by HBM)
template <int DT>
__global__ void __launch_bounds__(256)
silu_and_mul_kernel(uint16_t* out, const uint16_t* x, uint32_t rows, int d, FastDiv chunks, const int* valid_rows, int rpc, long row0) {
  const uint32_t total = live_rows(rows, valid_rows, rpc, row0) * chunks.d;
  for (uint32_t i = blockIdx.x * 256 + threadIdx.x; i < total; i += gridDim.x * 256) {
    const uint32_t r = chunks.div(i), c = i - r * chunks.d;
    const uint16_t* xr = x + (size_t)r * 2 * d + 8 * c;
    float a[8], b[8], y[8];
    unpack8<DT>(*(const u4*)xr, a);
    unpack8<DT>(*(const u4*)(xr + d), b);
    silu_mul8(a, b, y);
    *(u4*)(out + (size_t)r * d + 8 * c) = pack8<DT>(y);
  }
}

// ---- per-token-group fp8 quantisation (optionally fused behind SiLU-gate) ---
// A group of `gs` elements is handled by gs/8 adjacent lanes (gs in 64,128,256,512).
template <int DT, bool SILU>
__device__ __forceinline__ void group_fp8_quant(uint8_t* out, float* scales, const uint16_t* x, uint32_t total, int K, const FastDiv& chunks, int lpg,
                                                uint32_t first, uint32_t step) {
  const int lg = 31 - __clz(lpg);
  for (uint32_t i0 = first; i0 < total; i0 += step) {
    const uint32_t i = i0 + threadIdx.x;
    const bool live = i < total;
    const uint32_t r = live ? chunks.div(i) : 0, c = live ? i - r * chunks.d : 0;
    float y[8];
    if (SILU) {
      const uint16_t* xr = x + (size_t)r * 2 * K + 8 * c;
      float a[8], b[8];
      unpack8<DT>(*(const u4*)xr, a);
      unpack8<DT>(*(const u4*)(xr + K), b);
      // the unfused sequence stores the gate output in the activation dtype
      silu_mul8(a, b, y);
#pragma unroll
      for (int e = 0; e < 8; e += 2) round_act2<DT>(y[e], y[e + 1]);
    } else {
      unpack8<DT>(*(const u4*)(x + (size_t)r * K + 8 * c), y);
    }
    float mx = 0.f;
#pragma unroll
    for (int e = 0; e < 8; e += 2) mx = SILU ? max_abs2(mx, y[e], y[e + 1]) : fmaxf(fmaxf(mx, fabsf(y[e])), fabsf(y[e + 1]));
    if (!live) mx = 0.f;
    mx = lane_group_max(mx, lpg);
    const float s = fmaxf(mx, 1e-10f) / FP8_MAX;
    const SharedDivisor by_s(s);
    float q[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) q[e] = clamp448(by_s.div(y[e]));
    if (live) {
      *(u2*)(out + (size_t)r * K + 8 * c) = to_fp8x8(q);
      // (a row is a whole number of groups: the groups of the matrix count through)
      if ((c & (lpg - 1)) == 0) scales[i >> lg] = s;
    }
  }
}
template <int DT, bool SILU>
__global__ void __launch_bounds__(256)
group_fp8_quant_kernel(uint8_t* out, float* scales, const uint16_t* x, uint32_t rows, int K, FastDiv chunks, int lpg,
                       const int* valid_rows, int rpc, long row0) {
  const uint32_t total = live_rows(rows, valid_rows, rpc, row0) * chunks.d;     // 8-element pieces; lpg (a power of two <= 64) lanes per group
  group_fp8_quant<DT, SILU>(out, scales, x, total, K, chunks, lpg, blockIdx.x * 256, gridDim.x * 256);
}

// The two things that fp8 experts need before their first GEMM and that do not need each other, side by side: the first workgroup aligns
// the slots, the others quantise the rows.  (The alignment is one workgroup's latency, 6 us alone, the rows 5 at 256 x 7168.  us, the whole layer, two
// launches -> here: 43.4 -> 41.2, 91.0 -> 88.2, 260.4 -> 257.7, 1739.9 -> 1735.3.)
template <int DT, typename IdT>
__global__ void __launch_bounds__(ALIGN_WAVES * 64)
moe_align_fp8_quant_kernel(uint8_t* out, float* scales, const uint16_t* x, uint32_t total, int K, FastDiv chunks, const IdT* topk_ids, int numel,
                           int top, int E, int B, int* sorted_ids, int cap, int* expert_ids, int nblocks, int* npp) {
  extern __shared__ int sm[];
  if (blockIdx.x == 0) return moe_align_ids(topk_ids, numel, top, (const int*)nullptr, E, B, (const int*)nullptr, sorted_ids, cap, expert_ids, nblocks, npp, sm);
  group_fp8_quant<DT, false>(out, scales, x, total, K, chunks, 16, (blockIdx.x - 1) * (ALIGN_WAVES * 64), (gridDim.x - 1) * (ALIGN_WAVES * 64));
}

// ---- per-token fp8 (one workgroup per row) and static fp8 --------------------
// Bound by latency up to some hundred rows, by HBM above: the row is read once, P pieces of 16 bytes per lane with
// all loads in flight together, and quantised from registers.
template <int DT, int P>
__global__ void __launch_bounds__(1024)
token_fp8_quant_row_kernel(uint8_t* out, float* scales, const uint16_t* x, int K, const int* valid_rows) {
  const long row = blockIdx.x;
  if (valid_rows && row >= *valid_rows) return;
  __shared__ float red[16];
  const int chunks = K / 8, nt = blockDim.x;
  const uint16_t* xr = x + row * K;
  u4 v[P];
#pragma unroll
  for (int i = 0; i < P; ++i) {
    const int c = threadIdx.x + nt * i;
    v[i] = *(const u4*)(xr + 8 * (c < chunks ? c : 0));     // (past the end: the first piece again, for the maximum)
  }
  float mx = 0.f;
#pragma unroll
  for (int i = 0; i < P; ++i) {
    float y[8];
    unpack8<DT>(v[i], y);
#pragma unroll
    for (int e = 0; e < 8; ++e) mx = fmaxf(mx, fabsf(y[e]));
  }
  mx = block_max(mx, red);
  const RowFp8 q(mx);
  if (threadIdx.x == 0) scales[row] = q.scale;
#pragma unroll
  for (int i = 0; i < P; ++i) {
    const int c = threadIdx.x + nt * i;
    float y[8];
    unpack8<DT>(v[i], y);
    const u2 codes = q.codes(y);
    if (c < chunks) *(u2*)(out + row * K + 8 * c) = codes;
  }
}

// any row length and alignment, one element at a time
template <int DT>
__global__ void __launch_bounds__(256)
token_fp8_quant_kernel(uint8_t* out, float* scales, const uint16_t* x, int K, const int* valid_rows) {
  const long row = blockIdx.x;
  if (valid_rows && row >= *valid_rows) return;
  __shared__ float red[16];
  float mx = 0.f;
  for (int k = threadIdx.x; k < K; k += 256) mx = fmaxf(mx, fabsf(Elem<DT>::to_f32(x[row * K + k])));
  mx = block_max(mx, red);
  const float s = fmaxf(mx, 1e-10f) / FP8_MAX;
  if (threadIdx.x == 0) scales[row] = s;
  const SharedDivisor by_s(s);
  for (int k = threadIdx.x; k < K; k += 256) {
    const float y = clamp448(by_s.div(Elem<DT>::to_f32(x[row * K + k])));
    int w = __builtin_amdgcn_cvt_pk_fp8_f32(y, y, 0, false);
    out[row * K + k] = (uint8_t)(w & 0xff);
  }
}

template <int DT>
void launch_token_quant(long rows, int K, hipStream_t st, uint8_t* out, float* scales, const uint16_t* x, const int* valid_rows) {
  const RowShape s = row_shape(rows, K, (((uintptr_t)x & 15) | ((uintptr_t)out & 7)) == 0, device_cu_count());
  const dim3 grid((unsigned)rows), block(s.threads);
  switch (s.pieces) {
    case 1: hipLaunchKernelGGL((token_fp8_quant_row_kernel<DT, 1>), grid, block, 0, st, out, scales, x, K, valid_rows); break;
    case 2: hipLaunchKernelGGL((token_fp8_quant_row_kernel<DT, 2>), grid, block, 0, st, out, scales, x, K, valid_rows); break;
    case 4: hipLaunchKernelGGL((token_fp8_quant_row_kernel<DT, 4>), grid, block, 0, st, out, scales, x, K, valid_rows); break;
    case 8: hipLaunchKernelGGL((token_fp8_quant_row_kernel<DT, 8>), grid, block, 0, st, out, scales, x, K, valid_rows); break;
    default: hipLaunchKernelGGL((token_fp8_quant_kernel<DT>), grid, dim3(256), 0, st, out, scales, x, K, valid_rows); break;
  }
}

// FUSE: 0 = quantise x; 1 = silu(x[:, :K]) * x[:, K:] first; 2 = x[:, :K] * x[:, K:] first
template <int DT, int FUSE>
__global__ void __launch_bounds__(256)
static_fp8_quant_kernel(uint8_t* out, const uint16_t* x, const float* scale, long rows, int K,
                        const int* valid_rows, int rpc) {
  const long nrow = valid_rows ? min(rows, (long)max(0, *valid_rows) * rpc) : rows;
  const float s = *scale;
  if ((K & 7) == 0) {
    // 8 elements per lane and step: 16-byte loads, 8-byte stores
    const int chunks = K / 8;
    const long total = nrow * chunks;
    for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < total; i += (long)gridDim.x * 256) {
      const long r = i / chunks;
      const int c = (int)(i - r * chunks);
      float v[8];
      if (FUSE) {
        float l[8], g[8];
        unpack8<DT>(*(const u4*)(x + r * 2 * K + 8 * c), l);
        unpack8<DT>(*(const u4*)(x + r * 2 * K + K + 8 * c), g);
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = round_act<DT>(FUSE == 1 ? silu_mul(l[e], g[e]) : l[e] * g[e]);
      } else {
        unpack8<DT>(*(const u4*)(x + r * K + 8 * c), v);
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = clamp448(v[e] / s);
      *(u2*)(out + r * K + 8 * c) = to_fp8x8(v);
    }
    return;
  }
  const long total = nrow * K;
  for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < total; i += (long)gridDim.x * 256) {
    float v;
    if (FUSE) {
      const long r = i / K;
      const int c = (int)(i - r * K);
      const float l = Elem<DT>::to_f32(x[r * 2 * K + c]), g = Elem<DT>::to_f32(x[r * 2 * K + K + c]);
      v = round_act<DT>(FUSE == 1 ? silu_mul(l, g) : l * g);
    } else {
      v = Elem<DT>::to_f32(x[i]);
    }
    const float y = clamp448(v / s);
    int w = __builtin_amdgcn_cvt_pk_fp8_f32(y, y, 0, false);
    out[i] = (uint8_t)(w & 0xff);
  }
}

// ---- moe_sum: out[m, :] = sum_t in[m, t, :] in fp32 --------------------------
// IDS: without the slots whose id, id_step words apart, is outside [0, E).  Two slots are on their way at a time there: the ids are one more line
// to wait for, 0.4 us of a layer of 68 where a slot's row and id were waited for before the next one's.
template <int DT_IN, int DT_OUT, bool IDS>
__global__ void __launch_bounds__(256)
moe_sum_kernel(void* out, const uint16_t* in, uint32_t rows, int T, int K, FastDiv chunks, const int* valid_rows, long row0, const int32_t* ids, int id_step,
               uint32_t E) {
  const uint32_t total = live_rows(rows, valid_rows, 1, row0) * chunks.d;
  for (uint32_t i = blockIdx.x * 256 + threadIdx.x; i < total; i += gridDim.x * 256) {
    const long r = chunks.div(i);
    const int c = (int)(i - (uint32_t)r * chunks.d);
    float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    constexpr int U = IDS ? 2 : 1;
    for (int t = 0; t < T; t += U) {
      u4 x[U];
      int id[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const long slot = r * T + min(t + u, T - 1);
        x[u] = *(const u4*)(in + slot * K + 8 * c);
        if (IDS) id[u] = ids[slot * id_step];
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        float v[8];
        unpack8<DT_IN>(x[u], v);
        const uint32_t keep = !IDS ? 0xffffffffu : t + u < T ? slot_mask(id[u], E) : 0u;
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[e] += bitcast<float>(bitcast<uint32_t>(v[e]) & keep);
      }
    }
    if (DT_OUT == MI355Q_F32) {
      float* o = (float*)out + r * K + 8 * c;
      *(f4*)o = (f4){acc[0], acc[1], acc[2], acc[3]};
      *(f4*)(o + 4) = (f4){acc[4], acc[5], acc[6], acc[7]};
    } else {
      *(u4*)((uint16_t*)out + r * K + 8 * c) = pack8<DT_OUT == MI355Q_F32 ? MI355Q_F16 : DT_OUT>(acc);
    }
  }
}

// ---- RMS norm (+ residual add) (+ quantisation of the normalised row) -------
// One workgroup per row, two passes over it (the second one hits the L2):
//   z = x (+ residual, rounded to the activation type and written back to residual)
//   n = act(z * rsqrt(mean(z^2) + eps)),  o = act(n * weight)
// then QM 0: o; 1: e4m3fn(clamp(o / scale)); 2: e4m3fn per group of gs with its own scale
// absmax / 448; 3: int8 rne(o * act(1 / scale)) -- each exactly what the separate
// quantisation operator makes of the stored o.
template <int DT, bool ADD, int QM>
__global__ void __launch_bounds__(256)
rms_norm_kernel(void* out, float* out_scales, const uint16_t* x, uint16_t* residual, const uint16_t* weight,
                const float* scale, float eps, int K, int gs) {
  const long row = blockIdx.x;
  const int chunks = K / 8;
  const uint16_t* xr = x + row * K;
  uint16_t* rr = ADD ? residual + row * K : nullptr;
  __shared__ float red[4];
  float ss = 0.f;
  for (int c = threadIdx.x; c < chunks; c += 256) {
    float v[8];
    unpack8<DT>(*(const u4*)(xr + 8 * c), v);
    if (ADD) {
      float r[8];
      unpack8<DT>(*(const u4*)(rr + 8 * c), r);
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = round_act<DT>(v[e] + r[e]);
      *(u4*)(rr + 8 * c) = pack8<DT>(v);
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) ss += v[e] * v[e];
  }
  ss = wave_sum(ss);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ss;
  __syncthreads();
  ss = (red[0] + red[1]) + (red[2] + red[3]);
  const float rs = rsqrtf(ss / (float)K + eps);
  float qs = 1.f;
  if (QM == 1) qs = *scale;
  if (QM == 3) qs = round_act<DT>(1.0f / *scale);
  const int lpg = QM == 2 ? gs / 8 : 1;
  const int padded = (chunks + 255) / 256 * 256;       // every lane stays in the loop for the group shuffles
  for (int c0 = threadIdx.x; c0 < padded; c0 += 256) {
    const bool live = c0 < chunks;
    const int c = live ? c0 : 0;
    float v[8], w[8];
    // a thread re-reads only what it wrote itself in the first pass
    unpack8<DT>(*(const u4*)((ADD ? (const uint16_t*)rr : xr) + 8 * c), v);
    unpack8<DT>(*(const u4*)(weight + 8 * c), w);
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = round_act<DT>(round_act<DT>(v[e] * rs) * w[e]);
    if (QM == 0) {
      if (live) *(u4*)((uint16_t*)out + row * K + 8 * c) = pack8<DT>(v);
    } else if (QM == 1) {
      float q[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) q[e] = clamp448(v[e] / qs);
      if (live) *(u2*)((uint8_t*)out + row * K + 8 * c) = to_fp8x8(q);
    } else if (QM == 2) {
      float mx = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) mx = fmaxf(mx, fabsf(v[e]));
      if (!live) mx = 0.f;
      mx = lane_group_max(mx, lpg);
      const float sg = fmaxf(mx, 1e-10f) / FP8_MAX;
      const SharedDivisor by_sg(sg);
      float q[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) q[e] = clamp448(by_sg.div(v[e]));
      if (live) {
        *(u2*)((uint8_t*)out + row * K + 8 * c) = to_fp8x8(q);
        if ((c % lpg) == 0) out_scales[row * (K / gs) + c / lpg] = sg;
      }
    } else {
      float q[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) q[e] = v[e] * qs;
      if (live) *(u2*)((uint8_t*)out + row * K + 8 * c) = pack_s8x8(q);
    }
  }
}

// The same operator with the row (and the weight vector) loaded once, P pieces of 16 bytes per lane with all loads in
// flight together, and both passes run from registers -- the loop version above waits for one piece at a time and
// reads the row twice.  Same arithmetic per element; only the order in which the squares are added differs.
template <int DT, bool ADD, int QM, int P>
__global__ void __launch_bounds__(1024)
rms_norm_row_kernel(void* out, float* out_scales, const uint16_t* x, uint16_t* residual, const uint16_t* weight,
                    const float* scale, float eps, int K, int lpg) {
  const long row = blockIdx.x;
  const int chunks = K / 8, nt = blockDim.x;
  const uint16_t* xr = x + row * K;
  uint16_t* rr = ADD ? residual + row * K : nullptr;
  __shared__ float red[16];
  u4 xv[P], rv[P], wv[P];
  bool live[P];
#pragma unroll
  for (int i = 0; i < P; ++i) {
    const int c0 = threadIdx.x + nt * i;
    live[i] = c0 < chunks;
    const int c = live[i] ? c0 : 0;
    xv[i] = *(const u4*)(xr + 8 * c);
    if (ADD) rv[i] = *(const u4*)(rr + 8 * c);
    wv[i] = *(const u4*)(weight + 8 * c);
  }
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < P; ++i) {
    float v[8];
    unpack8<DT>(xv[i], v);
    if (ADD) {
      float r[8];
      unpack8<DT>(rv[i], r);
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = round_act<DT>(v[e] + r[e]);
      xv[i] = pack8<DT>(v);
      // (what follows starts from the stored 16-bit values in both variants: from known values the compiler takes other
      // instructions for the sum and the first rounding, and the operators would differ in the last place)
      asm("" : "+v"(xv[i]));
      if (live[i]) *(u4*)(rr + 8 * (threadIdx.x + nt * i)) = xv[i];
      unpack8<DT>(xv[i], v);
    }
    float s = ss;
#pragma unroll
    for (int e = 0; e < 8; ++e) s = __builtin_fmaf(v[e], v[e], s);
    ss = live[i] ? s : ss;
  }
  ss = block_sum(ss, red);
  const float rs = rsqrtf(ss / (float)K + eps);
  float qs = 1.f;
  if (QM == 1) qs = *scale;
  if (QM == 3) qs = round_act<DT>(1.0f / *scale);
#pragma unroll
  for (int i = 0; i < P; ++i) {
    const int c = threadIdx.x + nt * i;                 // (every lane stays for the group shuffles)
    float w[8], y[8];
    unpack8<DT>(xv[i], y);
    unpack8<DT>(wv[i], w);
#pragma unroll
    for (int e = 0; e < 8; e += 2) {
      y[e] *= rs, y[e + 1] *= rs;
      round_act2<DT>(y[e], y[e + 1]);
      y[e] *= w[e], y[e + 1] *= w[e + 1];
      round_act2<DT>(y[e], y[e + 1]);
    }
    if (QM == 0) {
      if (live[i]) *(u4*)((uint16_t*)out + row * K + 8 * c) = pack8<DT>(y);
    } else if (QM == 1) {
      float q[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) q[e] = clamp448(y[e] / qs);
      if (live[i]) *(u2*)((uint8_t*)out + row * K + 8 * c) = to_fp8x8(q);
    } else if (QM == 2) {
      float mx = 0.f;
#pragma unroll
      for (int e = 0; e < 8; e += 2) mx = max_abs2(mx, y[e], y[e + 1]);
      if (!live[i]) mx = 0.f;
      mx = lane_group_max(mx, lpg);
      const float sg = fmaxf(mx, 1e-10f) / FP8_MAX;
      const SharedDivisor by_sg(sg);
      float q[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) q[e] = clamp448(by_sg.div(y[e]));
      if (live[i]) {
        *(u2*)((uint8_t*)out + row * K + 8 * c) = to_fp8x8(q);
        if ((c & (lpg - 1)) == 0) out_scales[(row * chunks + c) >> (31 - __clz(lpg))] = sg;
      }
    } else {
      float q[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) q[e] = y[e] * qs;
      if (live[i]) *(u2*)((uint8_t*)out + row * K + 8 * c) = pack_s8x8(q);
    }
  }
}

template <int DT, bool ADD, int QM>
void launch_rms_mode(long rows, hipStream_t st, void* out, float* out_scales, const uint16_t* x, uint16_t* residual,
                     const uint16_t* weight, const float* scale, float eps, int K, int gs) {
  const dim3 grid((unsigned)rows);
  const RowShape s = row_shape(rows, K, true, device_cu_count());      // (the operator asks for 16-byte rows)
  const dim3 block(s.threads);
  const int lpg = QM == 2 ? gs / 8 : 1;
  switch (s.pieces) {
    case 1: hipLaunchKernelGGL((rms_norm_row_kernel<DT, ADD, QM, 1>), grid, block, 0, st, out, out_scales, x, residual, weight, scale, eps, K, lpg); break;
    case 2: hipLaunchKernelGGL((rms_norm_row_kernel<DT, ADD, QM, 2>), grid, block, 0, st, out, out_scales, x, residual, weight, scale, eps, K, lpg); break;
    case 4: hipLaunchKernelGGL((rms_norm_row_kernel<DT, ADD, QM, 4>), grid, block, 0, st, out, out_scales, x, residual, weight, scale, eps, K, lpg); break;
    default: hipLaunchKernelGGL((rms_norm_kernel<DT, ADD, QM>), grid, dim3(256), 0, st, out, out_scales, x, residual, weight, scale, eps, K, gs); break;
  }
}

template <int DT, bool ADD>
void launch_rms(int qm, long rows, hipStream_t st, void* out, float* out_scales, const uint16_t* x, uint16_t* residual,
                const uint16_t* weight, const float* scale, float eps, int K, int gs) {
  switch (qm) {
    case 0: launch_rms_mode<DT, ADD, 0>(rows, st, out, out_scales, x, residual, weight, scale, eps, K, gs); break;
    case 1: launch_rms_mode<DT, ADD, 1>(rows, st, out, out_scales, x, residual, weight, scale, eps, K, gs); break;
    case 2: launch_rms_mode<DT, ADD, 2>(rows, st, out, out_scales, x, residual, weight, scale, eps, K, gs); break;
    default: launch_rms_mode<DT, ADD, 3>(rows, st, out, out_scales, x, residual, weight, scale, eps, K, gs); break;
  }
}

// rows per launch of the kernels that index their 16-byte pieces with 31 bits
inline long rows_per_launch(int chunks) { return (long)0x7fff0000 / chunks; }

inline unsigned grid_for(long items) {
  long b = (items + 255) / 256;
  long cap = (long)device_cu_count() * 16;
  return (unsigned)(b < 1 ? 1 : (b > cap ? cap : b));
}

}  // namespace

// ids null: every slot counts
int moe_sum_launch(void* out, const void* in, long rows, int topk, int K, int in_dtype, int out_dtype, const int32_t* valid_rows, const int32_t* ids,
                   int id_step, int E, hipStream_t st) {
  MQ_REQUIRE(rows >= 0 && topk > 0 && K > 0 && K % 8 == 0, "moe_sum: bad shape rows=%ld topk=%d K=%d (K %% 8 == 0)", rows, topk, K);
  if (rows == 0) return 0;
  MQ_REQUIRE(out && in, "moe_sum: null pointer");
  MQ_REQUIRE(in_dtype == MI355Q_F16 || in_dtype == MI355Q_BF16, "moe_sum: input dtype %d must be f16 or bf16", in_dtype);
  MQ_REQUIRE(out_dtype == in_dtype || out_dtype == MI355Q_F32, "moe_sum: output dtype %d must equal the input's or be f32", out_dtype);
  MQ_REQUIRE(!ids || out_dtype == in_dtype, "moe_sum: with ids the output dtype %d must equal the input's", out_dtype);
  const FastDiv chunks((uint32_t)(K / 8));
  for (long r0 = 0; r0 < rows; r0 += rows_per_launch(K / 8)) {
    const uint32_t n = (uint32_t)std::min(rows - r0, rows_per_launch(K / 8));
    const unsigned g = grid_for((long)n * (K / 8));
    const uint16_t* p = (const uint16_t*)in + r0 * topk * K;
    void* o = (char*)out + r0 * K * (out_dtype == MI355Q_F32 ? 4 : 2);
    const int32_t* const id = ids ? ids + r0 * topk * id_step : nullptr;
#define MQ_SUM(IN, OUT, IDS) \
  hipLaunchKernelGGL((moe_sum_kernel<IN, OUT, IDS>), dim3(g), dim3(256), 0, st, o, p, n, topk, K, chunks, valid_rows, r0, id, id_step, (uint32_t)E)
    if (in_dtype == MI355Q_F16) {
      if (ids) MQ_SUM(MI355Q_F16, MI355Q_F16, true);
      else if (out_dtype == MI355Q_F16) MQ_SUM(MI355Q_F16, MI355Q_F16, false);
      else MQ_SUM(MI355Q_F16, MI355Q_F32, false);
    } else {
      if (ids) MQ_SUM(MI355Q_BF16, MI355Q_BF16, true);
      else if (out_dtype == MI355Q_BF16) MQ_SUM(MI355Q_BF16, MI355Q_BF16, false);
      else MQ_SUM(MI355Q_BF16, MI355Q_F32, false);
    }
#undef MQ_SUM
  }
  MQ_LAUNCH_CHECK("moe_sum");
  return 0;
}

}  // namespace mi355q

using namespace mi355q;

#define MQ_DISPATCH_16(dtype, CALL_F16, CALL_BF16, what)             \
  do {                                                               \
    if ((dtype) == MI355Q_F16) { CALL_F16; }                         \
    else if ((dtype) == MI355Q_BF16) { CALL_BF16; }                  \
    else MQ_REQUIRE(false, what ": dtype %d must be f16 or bf16", (int)(dtype)); \
  } while (0)

extern "C" int mi355q_silu_and_mul(void* out, const void* x, long rows, int d, int dtype,
                                   const int32_t* valid_rows, int rows_per_count, void* stream) {
  if (rows_per_count < 1) rows_per_count = 1;
  MQ_REQUIRE(rows >= 0 && d > 0 && d % 8 == 0, "silu_and_mul: bad shape rows=%ld d=%d (d %% 8 == 0)", rows, d);
  if (rows == 0) return 0;
  MQ_REQUIRE(out && x, "silu_and_mul: null pointer");
  MQ_REQUIRE(dtype == MI355Q_F16 || dtype == MI355Q_BF16, "silu_and_mul: dtype %d must be f16 or bf16", dtype);
  hipStream_t st = as_stream(stream);
  const FastDiv chunks((uint32_t)(d / 8));
  for (long r0 = 0; r0 < rows; r0 += rows_per_launch(d / 8)) {
    const uint32_t n = (uint32_t)std::min(rows - r0, rows_per_launch(d / 8));
    const unsigned g = grid_for((long)n * (d / 8));
    uint16_t* o = (uint16_t*)out + r0 * d;
    const uint16_t* xp = (const uint16_t*)x + r0 * 2 * d;
    if (dtype == MI355Q_F16)
      hipLaunchKernelGGL((silu_and_mul_kernel<MI355Q_F16>), dim3(g), dim3(256), 0, st, o, xp, n, d, chunks, valid_rows, rows_per_count, r0);
    else
      hipLaunchKernelGGL((silu_and_mul_kernel<MI355Q_BF16>), dim3(g), dim3(256), 0, st, o, xp, n, d, chunks, valid_rows, rows_per_count, r0);
  }
  MQ_LAUNCH_CHECK("silu_and_mul");
  return 0;
}

extern "C" int mi355q_fp8_group_quant(uint8_t* out, float* scales, const void* x, long rows, int K,
                                      int group_size, int fuse_silu_mul, int dtype,
                                      const int32_t* valid_rows, int rows_per_count, void* stream) {
  if (rows_per_count < 1) rows_per_count = 1;
  MQ_REQUIRE(rows >= 0 && K > 0, "fp8_group_quant: bad shape rows=%ld K=%d", rows, K);
  if (rows == 0) return 0;
  MQ_REQUIRE(out && scales && x, "fp8_group_quant: null pointer");
  MQ_REQUIRE(group_size == 64 || group_size == 128 || group_size == 256 || group_size == 512,
             "fp8_group_quant: group_size=%d must be 64, 128, 256 or 512", group_size);
  MQ_REQUIRE(K % group_size == 0, "fp8_group_quant: K=%d must be a multiple of group_size=%d", K, group_size);
  MQ_REQUIRE(dtype == MI355Q_F16 || dtype == MI355Q_BF16, "fp8_group_quant: dtype %d must be f16 or bf16", dtype);
  hipStream_t st = as_stream(stream);
  const FastDiv chunks((uint32_t)(K / 8));
  const int lpg = group_size / 8;
  const bool f16 = dtype == MI355Q_F16;
  for (long r0 = 0; r0 < rows; r0 += rows_per_launch(K / 8)) {
    const uint32_t n = (uint32_t)std::min(rows - r0, rows_per_launch(K / 8));
    // whole groups must sit inside one workgroup pass: 256 lanes cover 2048 elements
    const unsigned g = grid_for((long)n * (K / 8));
    uint8_t* o = out + r0 * K;
    float* sc = scales + r0 * (K / group_size);
    const uint16_t* xp = (const uint16_t*)x + r0 * K * (fuse_silu_mul ? 2 : 1);
    if (fuse_silu_mul && f16)
      hipLaunchKernelGGL((group_fp8_quant_kernel<MI355Q_F16, true>), dim3(g), dim3(256), 0, st, o, sc, xp, n, K, chunks, lpg, valid_rows, rows_per_count, r0);
    else if (fuse_silu_mul)
      hipLaunchKernelGGL((group_fp8_quant_kernel<MI355Q_BF16, true>), dim3(g), dim3(256), 0, st, o, sc, xp, n, K, chunks, lpg, valid_rows, rows_per_count, r0);
    else if (f16)
      hipLaunchKernelGGL((group_fp8_quant_kernel<MI355Q_F16, false>), dim3(g), dim3(256), 0, st, o, sc, xp, n, K, chunks, lpg, valid_rows, rows_per_count, r0);
    else
      hipLaunchKernelGGL((group_fp8_quant_kernel<MI355Q_BF16, false>), dim3(g), dim3(256), 0, st, o, sc, xp, n, K, chunks, lpg, valid_rows, rows_per_count, r0);
  }
  MQ_LAUNCH_CHECK("fp8_group_quant");
  return 0;
}

extern "C" int mi355q_fp8_token_quant(uint8_t* out, float* scales, const void* x, int rows, int K, int dtype,
                                      const int32_t* valid_rows, void* stream) {
  MQ_REQUIRE(rows >= 0 && K > 0, "fp8_token_quant: bad shape rows=%d K=%d", rows, K);
  if (rows == 0) return 0;
  MQ_REQUIRE(out && scales && x, "fp8_token_quant: null pointer");
  hipStream_t st = as_stream(stream);
  MQ_DISPATCH_16(dtype,
    launch_token_quant<MI355Q_F16>(rows, K, st, out, scales, (const uint16_t*)x, valid_rows),
    launch_token_quant<MI355Q_BF16>(rows, K, st, out, scales, (const uint16_t*)x, valid_rows),
    "fp8_token_quant");
  MQ_LAUNCH_CHECK("fp8_token_quant");
  return 0;
}

extern "C" int mi355q_fp8_static_quant(uint8_t* out, const void* x, const float* scale, long rows, int K,
                                       int fuse_silu_mul, int dtype, const int32_t* valid_rows,
                                       int rows_per_count, void* stream) {
  if (rows_per_count < 1) rows_per_count = 1;
  MQ_REQUIRE(rows >= 0 && K > 0, "fp8_static_quant: bad shape rows=%ld K=%d", rows, K);
  if (rows == 0) return 0;
  MQ_REQUIRE(out && scale && x, "fp8_static_quant: null pointer");
  hipStream_t st = as_stream(stream);
  unsigned g = grid_for((K & 7) == 0 ? rows * (K / 8) : rows * K);
  MQ_REQUIRE(fuse_silu_mul >= 0 && fuse_silu_mul <= 2, "fp8_static_quant: unknown fusion %d", fuse_silu_mul);
  if (fuse_silu_mul == 1) {
    MQ_DISPATCH_16(dtype,
      hipLaunchKernelGGL((static_fp8_quant_kernel<MI355Q_F16, 1>), dim3(g), dim3(256), 0, st, out, (const uint16_t*)x, scale, rows, K, valid_rows, rows_per_count),
      hipLaunchKernelGGL((static_fp8_quant_kernel<MI355Q_BF16, 1>), dim3(g), dim3(256), 0, st, out, (const uint16_t*)x, scale, rows, K, valid_rows, rows_per_count),
      "fp8_static_quant");
  } else if (fuse_silu_mul == 2) {
    MQ_DISPATCH_16(dtype,
      hipLaunchKernelGGL((static_fp8_quant_kernel<MI355Q_F16, 2>), dim3(g), dim3(256), 0, st, out, (const uint16_t*)x, scale, rows, K, valid_rows, rows_per_count),
      hipLaunchKernelGGL((static_fp8_quant_kernel<MI355Q_BF16, 2>), dim3(g), dim3(256), 0, st, out, (const uint16_t*)x, scale, rows, K, valid_rows, rows_per_count),
      "fp8_static_quant");
  } else {
    MQ_DISPATCH_16(dtype,
      hipLaunchKernelGGL((static_fp8_quant_kernel<MI355Q_F16, 0>), dim3(g), dim3(256), 0, st, out, (const uint16_t*)x, scale, rows, K, valid_rows, rows_per_count),
      hipLaunchKernelGGL((static_fp8_quant_kernel<MI355Q_BF16, 0>), dim3(g), dim3(256), 0, st, out, (const uint16_t*)x, scale, rows, K, valid_rows, rows_per_count),
      "fp8_static_quant");
  }
  MQ_LAUNCH_CHECK("fp8_static_quant");
  return 0;
}

extern "C" int mi355q_moe_sum(void* out, const void* in, long rows, int topk, int K, int in_dtype,
                              int out_dtype, const int32_t* valid_rows, void* stream) {
  return moe_sum_launch(out, in, rows, topk, K, in_dtype, out_dtype, valid_rows, nullptr, 1, 0, as_stream(stream));
}

// ---- fp8-e4m3fn -> f16 / bf16, exact (every e4m3fn value is representable in both) ----
template <int DT>
__global__ void __launch_bounds__(256)
fp8_to_half_kernel(uint16_t* out, const uint32_t* in, long words) {
  for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < words; i += (long)gridDim.x * 256) {
    const int w = (int)in[i];
    const f2 lo = __builtin_amdgcn_cvt_pk_f32_fp8(w, false), hi = __builtin_amdgcn_cvt_pk_f32_fp8(w, true);
    uint2 o;
    o.x = (uint32_t)Elem<DT>::from_f32(lo.x) | ((uint32_t)Elem<DT>::from_f32(lo.y) << 16);
    o.y = (uint32_t)Elem<DT>::from_f32(hi.x) | ((uint32_t)Elem<DT>::from_f32(hi.y) << 16);
    *(uint2*)(out + 4 * i) = o;
  }
}

extern "C" int mi355q_fp8_to_half(void* out, const uint8_t* in, long n, int out_dtype, void* stream) {
  MQ_REQUIRE(n >= 0 && n % 4 == 0, "fp8_to_half: element count %ld must be a multiple of 4", n);
  if (n == 0) return 0;
  MQ_REQUIRE(out && in, "fp8_to_half: null pointer");
  MQ_REQUIRE(out_dtype == MI355Q_F16 || out_dtype == MI355Q_BF16, "fp8_to_half: output dtype %d must be f16 or bf16", out_dtype);
  hipStream_t st = as_stream(stream);
  const unsigned g = grid_for(n / 4);
  if (out_dtype == MI355Q_F16)
    hipLaunchKernelGGL((fp8_to_half_kernel<MI355Q_F16>), dim3(g), dim3(256), 0, st, (uint16_t*)out, (const uint32_t*)in, n / 4);
  else
    hipLaunchKernelGGL((fp8_to_half_kernel<MI355Q_BF16>), dim3(g), dim3(256), 0, st, (uint16_t*)out, (const uint32_t*)in, n / 4);
  MQ_LAUNCH_CHECK("fp8_to_half");
  return 0;
}

extern "C" int mi355q_rms_norm(void* out, float* out_scales, const void* x, void* residual, const void* weight,
                               const float* scale, float eps, long rows, int K, int quant_mode, int group_size,
                               int dtype, void* stream) {
  MQ_REQUIRE(rows >= 0 && K > 0 && K % 8 == 0, "rms_norm: bad shape rows=%ld K=%d (K %% 8 == 0)", rows, K);
  if (rows == 0) return 0;
  MQ_REQUIRE(out && x && weight, "rms_norm: null pointer");
  MQ_REQUIRE(rows <= 0x7fffffffL, "rms_norm: too many rows");
  MQ_REQUIRE(quant_mode >= 0 && quant_mode <= 3, "rms_norm: quant_mode %d must be 0..3", quant_mode);
  MQ_REQUIRE(dtype == MI355Q_F16 || dtype == MI355Q_BF16, "rms_norm: dtype %d must be f16 or bf16", dtype);
  if (quant_mode == 1 || quant_mode == 3) MQ_REQUIRE(scale, "rms_norm: static scale missing");
  if (quant_mode == 2) {
    MQ_REQUIRE(out_scales, "rms_norm: group scales output missing");
    MQ_REQUIRE((group_size == 64 || group_size == 128 || group_size == 256 || group_size == 512) && K % group_size == 0,
               "rms_norm: group_size %d must be 64..512 (a power of two) and divide K=%d", group_size, K);
  }
  hipStream_t st = as_stream(stream);
  const long grid = rows;
  const uint16_t* xp = (const uint16_t*)x;
  uint16_t* rp = (uint16_t*)residual;
  const uint16_t* wp = (const uint16_t*)weight;
  if (dtype == MI355Q_F16) {
    if (residual) launch_rms<MI355Q_F16, true>(quant_mode, grid, st, out, out_scales, xp, rp, wp, scale, eps, K, group_size);
    else launch_rms<MI355Q_F16, false>(quant_mode, grid, st, out, out_scales, xp, rp, wp, scale, eps, K, group_size);
  } else {
    if (residual) launch_rms<MI355Q_BF16, true>(quant_mode, grid, st, out, out_scales, xp, rp, wp, scale, eps, K, group_size);
    else launch_rms<MI355Q_BF16, false>(quant_mode, grid, st, out, out_scales, xp, rp, wp, scale, eps, K, group_size);
  }
  MQ_LAUNCH_CHECK("rms_norm");
  return 0;
}

extern "C" int mi355q_moe_align_fp8_quant(uint8_t* q, float* q_scales, const void* x, long rows, int K, int dtype, const void* topk_ids,
                                          int ids_are_int64, int numel, int topk, int num_experts, int block_size, int32_t* sorted_token_ids,
                                          int32_t* expert_ids, int32_t* num_tokens_post_pad, void* stream) {
  MQ_REQUIRE(rows > 0 && K > 0 && K % 128 == 0 && numel > 0 && num_experts > 0 && block_size > 0 && topk > 0,
             "moe_align_fp8_quant: bad arguments rows=%ld K=%d numel=%d E=%d block=%d topk=%d", rows, K, numel, num_experts, block_size, topk);
  MQ_REQUIRE(q && q_scales && x && topk_ids && sorted_token_ids && expert_ids && num_tokens_post_pad, "moe_align_fp8_quant: null pointer");
  MQ_REQUIRE(dtype == MI355Q_F16 || dtype == MI355Q_BF16, "moe_align_fp8_quant: dtype %d must be f16 or bf16", dtype);
  const size_t shmem = moe_align_lds(num_experts);
  if (rows > rows_per_launch(K / 8) || shmem > 64 * 1024 || num_experts > 1024) {      // (refused there, or too many rows for one launch)
    if (int rc = mi355q_fp8_group_quant(q, q_scales, x, rows, K, 128, 0, dtype, nullptr, 1, stream)) return rc;
    return mi355q_moe_align_block_size(topk_ids, ids_are_int64, numel, topk, nullptr, num_experts, block_size, nullptr, sorted_token_ids, expert_ids,
                                       num_tokens_post_pad, stream);
  }
  const uint32_t total = (uint32_t)rows * (uint32_t)(K / 8);
  const unsigned grid = 1 + (unsigned)std::min<long>(((long)total + 1023) / 1024, (long)device_cu_count() * 8);
  const int cap = numel + num_experts * (block_size - 1);
  const FastDiv chunks((uint32_t)(K / 8));
#define MQ_FRONT(DT, ID)                                                                                                                    \
  hipLaunchKernelGGL((moe_align_fp8_quant_kernel<DT, ID>), dim3(grid), dim3(ALIGN_WAVES * 64), shmem, as_stream(stream), q, q_scales,          \
                     (const uint16_t*)x, total, K, chunks, (const ID*)topk_ids, numel, topk, num_experts, block_size, sorted_token_ids, cap,    \
                     expert_ids, cap / block_size, num_tokens_post_pad)
  if (dtype == MI355Q_F16 && ids_are_int64) MQ_FRONT(MI355Q_F16, long);
  else if (dtype == MI355Q_F16) MQ_FRONT(MI355Q_F16, int);
  else if (ids_are_int64) MQ_FRONT(MI355Q_BF16, long);
  else MQ_FRONT(MI355Q_BF16, int);
#undef MQ_FRONT
  MQ_LAUNCH_CHECK("moe_align_fp8_quant");
  return 0;
}
