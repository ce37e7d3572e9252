// Shared helpers for the gfx950 kernels: error reporting, vector types,
// small device utilities.  Everything here is internal to the library.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdio.h>
#include <stdarg.h>

#include "../../include/mi355q.h"

namespace mi355q {

// ---- host-side error plumbing ---------------------------------------------
void set_error(const char* fmt, ...);

#define MQ_REQUIRE(cond, ...)                 \
  do {                                        \
    if (!(cond)) {                            \
      ::mi355q::set_error(__VA_ARGS__);       \
      return 1;                               \
    }                                         \
  } while (0)

#define MQ_LAUNCH_CHECK(what)                                              \
  do {                                                                     \
    hipError_t e__ = hipGetLastError();                                    \
    if (e__ != hipSuccess) {                                               \
      ::mi355q::set_error("%s: launch failed: %s", what,                   \
                          hipGetErrorString(e__));                         \
      return 2;                                                            \
    }                                                                      \
  } while (0)

// ---- vector types ----------------------------------------------------------
typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef _Float16 h4 __attribute__((ext_vector_type(4)));
typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef __bf16 b8 __attribute__((ext_vector_type(8)));
typedef short s8v __attribute__((ext_vector_type(8)));
typedef float f2 __attribute__((ext_vector_type(2)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef float f16v __attribute__((ext_vector_type(16)));
typedef int i4 __attribute__((ext_vector_type(4)));
typedef int i8v __attribute__((ext_vector_type(8)));
typedef int i16v __attribute__((ext_vector_type(16)));
typedef uint32_t u2 __attribute__((ext_vector_type(2)));
typedef uint32_t u4 __attribute__((ext_vector_type(4)));

template <typename T, typename U>
__device__ __forceinline__ T bitcast(const U& u) {
  static_assert(sizeof(T) == sizeof(U), "bitcast size");
  return __builtin_bit_cast(T, u);
}

// bf16 -> f32 is a shift; f32 -> bf16 is the hardware conversion of gfx950 (v_cvt_pk_bf16_f32:
// round to nearest even, NaN stays NaN), one instruction where the bit manipulation took six
__device__ __forceinline__ float bf16_to_f32(uint16_t v) {
  return bitcast<float>((uint32_t)v << 16);
}
__device__ __forceinline__ uint16_t f32_to_bf16(float f) {
  return bitcast<uint16_t>((__bf16)f);
}

// Epilogue of the scaled integer / fp8 GEMMs, (sum * x_scale) * w_scale (+ bias), with every operation
// rounded on its own: left to the compiler's contraction rules the multiply-add pairs fuse in some
// kernels (and in some paths of one kernel) and not in others, and kernels that must agree bit for bit
// -- the tile kernels, the weight-streaming kernels, the split-K epilogue -- would differ in the last place.
__device__ __forceinline__ float scaled_sum(float sum, float x_scale, float w_scale) {
#pragma clang fp contract(off)
  const float t = sum * x_scale;
  return t * w_scale;
}
__device__ __forceinline__ float plus_bias(float v, float bias) {
#pragma clang fp contract(off)
  return v + bias;
}

template <int DT> struct Elem;            // activation element traits
template <> struct Elem<MI355Q_F16> {
  typedef _Float16 type;
  static __device__ __forceinline__ float to_f32(uint16_t raw) {
    return (float)bitcast<_Float16>(raw);
  }
  static __device__ __forceinline__ uint16_t from_f32(float f) {
    return bitcast<uint16_t>((_Float16)f);
  }
};
template <> struct Elem<MI355Q_BF16> {
  typedef __bf16 type;
  static __device__ __forceinline__ float to_f32(uint16_t raw) { return bf16_to_f32(raw); }
  static __device__ __forceinline__ uint16_t from_f32(float f) { return f32_to_bf16(f); }
};

// A pre-scaled zero-point zs (16 bits, as stored) of a group with scale s, for kernels whose operands are q - z with an integer
// z: w = q s - zs is (q - z) s - rest.  Where zs is bit for bit an integer 0 .. 15 times s, as the loaders that pre-multiply make
// it, rest is 0 (zs read before its rounding); any other zs is taken as given.  A scale of 0 has w = -zs.
template <int DT>
__device__ __forceinline__ float prescaled_zero(uint16_t zs, float s) {
  return fminf(fmaxf(__builtin_rintf(Elem<DT>::to_f32(zs) / s), 0.0f), 15.0f);     // (0 / 0: 0)
}
// not 0: z times s is not zs (what the loops look at; the rest itself only where there is one)
template <int DT>
__device__ __forceinline__ uint32_t prescaled_differs(uint16_t zs, float z, float s) { return Elem<DT>::from_f32(z * s) ^ zs; }
template <int DT>
__device__ __forceinline__ float prescaled_rest(uint16_t zs, float s) {
  const float z = prescaled_zero<DT>(zs, s), zf = Elem<DT>::to_f32(zs);
  return z == 0.0f ? zf : prescaled_differs<DT>(zs, z, s) ? __builtin_fmaf(-z, s, zf) : 0.0f;
}

// Kernels whose accumulators alone fill 128+ registers call this once: an
// inline-asm AGPR operand makes the compiler keep MFMA accumulators in the
// accumulation half of the register file (AGPR-form MFMA) instead of using it
// only as a spill area for VGPR-form MFMAs.
__device__ __forceinline__ void use_agpr_accumulators() {
  int t = 0;
  asm volatile("" : "+a"(t));
}

// Buffer loads: an offset at or past the descriptor's size reads as zero
// without touching memory, which makes "no such K block" a branch-free case
// (callers add 2^31 to the lane offset; every buffer here is below 2 GiB).
typedef __amdgpu_buffer_rsrc_t rsrc_t;
__device__ __forceinline__ rsrc_t make_rsrc(const void* p, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (int)bytes, 0x00020000);
}
__device__ __forceinline__ u4 buf_load16(rsrc_t r, uint32_t off) {
  return bitcast<u4>(__builtin_amdgcn_raw_buffer_load_b128(r, (int)off, 0, 0));
}
// streamed once: non-temporal
__device__ __forceinline__ u4 buf_load16_nt(rsrc_t r, uint32_t off) {
  return bitcast<u4>(__builtin_amdgcn_raw_buffer_load_b128(r, (int)off, 0, 2));
}

// Copies straight from global memory into LDS, 64 lanes x 16 (or 4) bytes, no registers between: lane l lands at the
// wavefront's LDS base + 16 l (4 l).  dma16 is the compiler's form, from an address per lane.  The others are inline
// assembly, from a 32-bit byte offset per lane and a base per wavefront: the compiler does not see them, places its waits
// for the LDS reads alone, and the kernel waits for the copies by hand (vmcnt).
__device__ __forceinline__ void dma16(const void* gptr, void* lds_wave_base) {
  __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)gptr,
                                   (__attribute__((address_space(3))) void*)lds_wave_base, 16, 0, 0);
}
__device__ __forceinline__ void lds_copy16(uint32_t voff, const void* sbase, uint32_t lds_addr) {
  // (uniform by construction; inside a divergent region the compiler may otherwise keep it in a vector register)
  lds_addr = __builtin_amdgcn_readfirstlane(lds_addr);
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"(voff), "s"(sbase), "s"(lds_addr) : "memory");
}
__device__ __forceinline__ void lds_copy4(uint32_t voff, const void* sbase, uint32_t lds_addr) {
  lds_addr = __builtin_amdgcn_readfirstlane(lds_addr);
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dword %0, %1" : : "v"(voff), "s"(sbase), "s"(lds_addr) : "memory");
}
// to lds_addr + more, both in scalar registers already
__device__ __forceinline__ void lds_copy16(uint32_t voff, const void* sbase, uint32_t lds_addr, uint32_t more) {
  asm volatile("s_add_u32 m0, %2, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"(voff), "s"(sbase), "s"(lds_addr), "s"(more) : "memory", "scc");
}
__device__ __forceinline__ void lds_copy4(uint32_t voff, const void* sbase, uint32_t lds_addr, uint32_t more) {
  asm volatile("s_add_u32 m0, %2, %3\n\ts_nop 0\n\tglobal_load_lds_dword %0, %1" : : "v"(voff), "s"(sbase), "s"(lds_addr), "s"(more) : "memory", "scc");
}
template <int OFF>
__device__ __forceinline__ void lds_copy16_next(uint32_t voff, const void* sbase) {   // the m0 of the copy before; OFF counts on both sides
  asm volatile("global_load_lds_dwordx4 %0, %1 offset:%2" : : "v"(voff), "s"(sbase), "n"(OFF) : "memory");
}

// Workgroups go to the eight XCDs in turn: XCD x takes the x-th eighth of the tiles (ordered by column), so that the row tiles
// of a column tile share one L2 and its weights pass it once, whatever the number of column tiles.  Column tiles that are parts of one
// block of the weights' layout (8 KiB of a slab or of a kslab group) belong on one XCD for the same reason: dealt out in turn, eight L2s take
// pieces of 1 .. 4 KiB out of every block, with its scales (us at one row, weights out of the caches, in turn -> here: int8 8192 x 8192 16.1 -> 12.7,
// 8192 x 10240 21.5 -> 18.6, 4096 x 4096 6.0 -> 5.4; W4A16 4096 x 6144 5.9 -> 5.3, 8192 x 8192 at 1 9.7 -> 8.9; a layer of 64 experts of
// 2048 x 2048, six to a token, at 4 tokens 31.0 -> 29.2).
__device__ __forceinline__ int xcd_tile() {
  const int share = (int)gridDim.x >> 3, odd = gridDim.x & 7, x8 = blockIdx.x & 7;
  return x8 * share + min(x8, odd) + ((int)blockIdx.x >> 3);
}

// Wavefront reductions on the data-parallel-primitive path (lane shifts inside the vector ALU, no trip
// through the LDS crossbar).  Every lane of the wavefront must be active.
// Whole wavefront: an inclusive scan within each row of 16 lanes (shifts by 1, 2, 4, 8; lanes a shift
// does not reach keep the identity), then lane 15 of rows 0 and 2 joins rows 1 and 3, lane 31 joins
// rows 2 and 3, and lane 63 holds the result, which is read back as a scalar.
#define MQ_DPP_REDUCE(v, ident, OP)                                                                     \
  do {                                                                                                  \
    v = OP(v, __builtin_amdgcn_update_dpp(ident, v, 0x111, 0xf, 0xf, false)); /* row_shr:1 */           \
    v = OP(v, __builtin_amdgcn_update_dpp(ident, v, 0x112, 0xf, 0xf, false)); /* row_shr:2 */           \
    v = OP(v, __builtin_amdgcn_update_dpp(ident, v, 0x114, 0xf, 0xf, false)); /* row_shr:4 */           \
    v = OP(v, __builtin_amdgcn_update_dpp(ident, v, 0x118, 0xf, 0xf, false)); /* row_shr:8 */           \
    v = OP(v, __builtin_amdgcn_update_dpp(ident, v, 0x142, 0xa, 0xf, false)); /* row_bcast:15 */        \
    v = OP(v, __builtin_amdgcn_update_dpp(ident, v, 0x143, 0xc, 0xf, false)); /* row_bcast:31 */        \
    v = __builtin_amdgcn_readlane(v, 63);                                                               \
  } while (0)
__device__ __forceinline__ int op_fmax_bits(int a, int b) { return __float_as_int(fmaxf(__int_as_float(a), __int_as_float(b))); }
__device__ __forceinline__ int op_fadd_bits(int a, int b) { return __float_as_int(__int_as_float(a) + __int_as_float(b)); }
__device__ __forceinline__ int op_imin(int a, int b) { return a < b ? a : b; }
__device__ __forceinline__ float wave_max(float x) {
  int v = __float_as_int(x);
  MQ_DPP_REDUCE(v, (int)0xff800000, op_fmax_bits);   // identity: -inf
  return __int_as_float(v);
}
__device__ __forceinline__ float wave_sum(float x) {
  int v = __float_as_int(x);
  MQ_DPP_REDUCE(v, 0, op_fadd_bits);
  return __int_as_float(v);
}
// max of values of at least 0 (no NaN) over aligned groups of `lanes` lanes (a power of two, 2 .. 64), the result in every lane of the
// group: swaps inside quads, mirrors of the half row and of the row of 16 lanes, LDS shuffles only
// for what crosses rows.  (As integers, which order such floats alike: an instruction a step.)
__device__ __forceinline__ float lane_group_max(float x, int lanes) {
  int v = __float_as_int(x);
  if (lanes >= 2) v = max(v, __builtin_amdgcn_update_dpp(v, v, 0xB1, 0xf, 0xf, false));             // quad_perm [1,0,3,2]
  if (lanes >= 4) v = max(v, __builtin_amdgcn_update_dpp(v, v, 0x4E, 0xf, 0xf, false));             // quad_perm [2,3,0,1]
  if (lanes >= 8) v = max(v, __builtin_amdgcn_update_dpp(v, v, 0x141, 0xf, 0xf, false));            // row_half_mirror
  if (lanes >= 16) {
    v = max(v, __builtin_amdgcn_update_dpp(v, v, 0x140, 0xf, 0xf, false));                          // row_mirror
    for (int o = 16; o < lanes; o <<= 1) v = max(v, __shfl_xor(v, o));
  }
  return __int_as_float(v);
}

// Fused-MoE grouped GEMMs: a block whose expert id lies outside [0, E) -- a non-local expert under an
// expert map, -1 in the reference (vllm_gcu/kernels/fused_moe.py:70-71, 106-107) -- contributes
// nothing.  Its workgroups read no weights and zero the columns [col0, col0 + ncols) (ncols % 4 == 0)
// of every valid slot row of the block; `ids` are the block's `rows` slot ids, pads >= numel.
__device__ __forceinline__ void zero_block_columns(uint16_t* out, const int* ids, int rows, int numel, int N,
                                                   int col0, int ncols, int nthreads) {
  const int per_row = ncols >> 2;
  for (int i = threadIdx.x; i < rows * per_row; i += nthreads) {
    const int r = i / per_row, piece = i - r * per_row;
    const int id = ids[r];
    if (id < numel) *(uint2*)(out + (size_t)id * N + col0 + 4 * piece) = make_uint2(0u, 0u);
  }
}

// n / d for a divisor known on the host and n < 2^31: a multiplication and two shifts, where the hardware-less 32- and
// 64-bit divisions of a kernel's index arithmetic take 30 .. 100 instructions
struct FastDiv {
  uint32_t d, mul, shift;
  FastDiv() = default;
  explicit FastDiv(uint32_t div) : d(div) {
    shift = 0;
    while (shift < 31 && (1u << shift) < div) ++shift;                      // 2^shift >= d
    mul = (uint32_t)(((uint64_t)1 << 32) * (((uint64_t)1 << shift) - div) / div + 1);
  }
  __device__ __forceinline__ uint32_t div(uint32_t n) const { return (__umulhi(n, mul) + n) >> shift; }
};

__device__ __forceinline__ float silu_mul(float a, float b) {
  return a * (1.0f / (1.0f + expf(-a))) * b;      // left * sigmoid(left) * right
}

// An estimate and its Newton step: the correctly rounded reciprocal of every float from 1 to 2^126, in three instructions where the division takes ten
__device__ __forceinline__ float short_reciprocal(float s) {
  const float y = __builtin_amdgcn_rcpf(s);
  return __builtin_fmaf(__builtin_fmaf(-s, y, 1.0f), y, y);
}
// ... of eight of each, to the same bits for every gate and up value of 16 bits; gates below -87, whose reciprocal is no normal number, take the division.  (This and the
// codes below are compared with the plain forms over all operands, csrc/bench/arith.hip.)
__device__ __forceinline__ void silu_mul8(const float* a, const float* b, float* y) {
  float s[8], r[8], m = 1.0f;
#pragma unroll
  for (int e = 0; e < 8; ++e) s[e] = 1.0f + expf(-a[e]);
#pragma unroll
  for (int e = 0; e < 8; ++e) m = fmaxf(m, s[e]);
  if (__any(m > 0x1p126f)) {
#pragma unroll
    for (int e = 0; e < 8; ++e) r[e] = 1.0f / s[e];
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e) r[e] = short_reciprocal(s[e]);
  }
  // (here, so that the last product is rounded to fp16 at once, as the single ones are)
#pragma unroll
  for (int e = 0; e < 8; ++e) y[e] = a[e] * r[e] * b[e];
}

// what silu_and_mul stores for a gate and an up column that are 16 bits already
template <int DT>
__device__ __forceinline__ uint16_t silu_mul16(uint16_t gate, uint16_t up) {
  if constexpr (DT == MI355Q_F16) {
    uint32_t h;                                      // (its product with the up column is rounded to fp16 at once)
    asm("v_fma_mixlo_f16 %0, %1, %2, 0 op_sel_hi:[0,1,0]" : "=v"(h) : "v"(silu_mul(Elem<DT>::to_f32(gate), 1.0f)), "v"((uint32_t)up));
    return (uint16_t)h;
  } else {
    return Elem<DT>::from_f32(silu_mul(Elem<DT>::to_f32(gate), Elem<DT>::to_f32(up)));
  }
}
template <int DT>
__device__ __forceinline__ uint32_t silu_mul16x2(uint32_t gate, uint32_t up) {
  return (uint32_t)silu_mul16<DT>((uint16_t)gate, (uint16_t)up) | ((uint32_t)silu_mul16<DT>((uint16_t)(gate >> 16), (uint16_t)(up >> 16)) << 16);
}

// all ones for a slot of one of the E experts, zero for one that no block holds (no comparison: behind a branch the slot's sums would be asked for
// only when its id has arrived)
__device__ __forceinline__ uint32_t slot_mask(int32_t id, int32_t E) {
  return (uint32_t)((id - E) & ~id) >> 31 ? 0xffffffffu : 0u;
}

constexpr float FP8_MAX = 448.0f;
template <int DT>
__device__ __forceinline__ float round_act(float f) {
  return Elem<DT>::to_f32(Elem<DT>::from_f32(f));
}

__device__ __forceinline__ float clamp448(float y) { return fminf(fmaxf(y, -FP8_MAX), FP8_MAX); }

// Two values rounded to the activation type (bf16: one conversion for both, which the compiler would take apart again).
template <int DT>
__device__ __forceinline__ void round_act2(float& a, float& b) {
  if constexpr (DT == MI355Q_BF16) {
    uint32_t v;
    asm("v_cvt_pk_bf16_f32 %0, %1, %2" : "=v"(v) : "v"(a), "v"(b));
    a = bitcast<float>(v << 16);
    b = bitcast<float>(v & 0xffff0000u);
  } else {
    a = round_act<DT>(a);
    b = round_act<DT>(b);
  }
}

// max(m, |a|, |b|) without the operands' NaNs, of results of arithmetic or conversions.  (In one instruction: fmaxf of values whose bits were
// moved about makes the compiler quiet NaNs first, which those results never need.)
__device__ __forceinline__ float max_abs2(float m, float a, float b) {
  float r;
  asm("v_max3_f32 %0, |%1|, |%2|, %3" : "=v"(r) : "v"(a), "v"(b), "v"(m));
  return r;
}

// a / s for many a and one s, with the result of the IEEE division, for what the quantisers divide: a of 16 bits, s = max(largest |a|, 1e-10) / 448.
// The correctly rounded reciprocal is made once per divisor (an estimate and its Newton step), per dividend the quotient estimate and its
// correction by the exact residual.  s is normal and |a / s| <= 448; a residual can only underflow where the quotient is far below the smallest fp8 step.  (One
// correction is enough: every pair of finite 16-bit values gives the division's fp8 code.)  An infinite s, of a group with an
// infinity, makes zeros of what is finite and NaN of the infinities; the residual is taken as s q - a, whose zero leaves the sign of a zero quotient alone.
struct SharedDivisor {
  float s, y;
  __device__ __forceinline__ explicit SharedDivisor(float s_) {
    const bool finite = s_ < __builtin_inff();
    s = finite ? s_ : 0.0f;
    y = finite ? short_reciprocal(s_) : 0.0f;
  }
  __device__ __forceinline__ float div(float a) const {
    const float q = a * y;
    return __builtin_fmaf(-__builtin_fmaf(q, s, -a), y, q);
  }
};

// Launch shape of the kernels that hold one row of K elements of 16 bits in registers (8 per lane and piece) between
// two passes over it: threads per row and pieces per lane.  Four pieces per lane at most where there are rows
// enough to fill the chip; with fewer rows than that a row is spread over more wavefronts, because the launch then
// takes as long as one row does.  pieces == 0: the row is too long, not a whole number of pieces or not aligned.
struct RowShape {
  int threads, pieces;
};
inline RowShape row_shape(long rows, int K, bool aligned, int cus) {
  const int chunks = K / 8;
  if (!aligned || K % 8 != 0 || chunks > 8 * 1024) return {256, 0};
  const int most = rows >= 4L * cus ? 4 : rows >= 2L * cus ? 2 : 1;
  int threads = 256;
  while (threads < 1024 && chunks > threads * most) threads *= 2;
  const int p = (chunks + threads - 1) / threads;
  return {threads, p <= 1 ? 1 : p <= 2 ? 2 : p <= 4 ? 4 : 8};
}
__device__ __forceinline__ float block_sum(float x, float* red) {
  x = wave_sum(x);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = x;
  __syncthreads();
  float s = red[0] + red[1];
  const int n = (int)(blockDim.x >> 6);                                    // 4, 8 or 16 wavefronts
  for (int i = 2; i < n; i += 2) s += red[i] + red[i + 1];
  return s;
}
// maximum over the workgroup (up to 16 wavefronts, all lanes active); `red` is 16 floats of LDS
__device__ __forceinline__ float block_max(float x, float* red) {
  x = wave_max(x);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = x;
  __syncthreads();
  float m = red[0];
  for (int i = 1; i < (int)(blockDim.x >> 6); ++i) m = fmaxf(m, red[i]);
  return m;
}

inline hipStream_t as_stream(void* s) { return reinterpret_cast<hipStream_t>(s); }

int device_cu_count();

// The order of the output tiles of a GEMM: K ranges, groups of row tiles, columns, row tiles of the group.  Workgroups go to the eight
// XCDs in turn; XCD x takes the x-th eighth of the tiles in this order, so that what it multiplies at a time is a block of few
// rows and few columns, which its L2 takes in once.  (Tile ids in steps of eight give an XCD nearly all rows and all columns, unless the
// columns or the row tiles are a multiple of eight.)
struct TileOrder {
  FastDiv range, group, rows, last;     // by the tiles of a K range and of a group, by the row tiles of a group and of the last one
  int mtiles, total;
  __device__ __forceinline__ void locate(int tile, int& tm, int& tn, int& split) const {
    const int x = tile & 7;
    uint32_t t = (uint32_t)(x * (total >> 3) + min(x, total & 7) + (tile >> 3));
    split = (int)range.div(t);
    t -= (uint32_t)split * range.d;
    const int g = (int)group.div(t), first = g * (int)rows.d;
    t -= (uint32_t)g * group.d;
    const bool whole = first + (int)rows.d <= mtiles;
    tn = (int)(whole ? rows.div(t) : last.div(t));
    tm = first + (int)t - tn * (int)(whole ? rows.d : last.d);
  }
};
// Row tiles of a group: those for which an XCD's L2 takes in the fewest bytes.  An XCD has an eighth of the tiles, as many at a time as
// its CUs hold; the tiles of a column want its weights once, and all columns share the rows of the group, which stay in the L2
// between rounds as far as they fit.  Weights that the last-level cache does not hold count twice (fp8 K 8192 x N 28672 at 1537 rows: one
// group of seven row tiles 327 us, two 338).  row_bytes, col_bytes: of a row tile and of a column tile over a K range.
inline TileOrder tile_order(int mtiles, int ntiles, int ranges, double row_bytes, double col_bytes, int per_cu = 1) {
  const double share = (double)mtiles * ntiles * ranges / 8, at_once = per_cu * device_cu_count() / 8.0;
  const double rounds = share > at_once ? share / at_once : 1.0, column = col_bytes * (col_bytes * ntiles * ranges > 1.6e8 ? 2 : 1);
  int rows = mtiles;
  double best = 1e30;
  for (int groups = 1; groups <= mtiles && groups <= 32; ++groups) {
    const int r = (mtiles + groups - 1) / groups;
    const bool astride = groups > 1 && (mtiles % groups != 0 || 8 % (groups * ranges) != 0);      // an XCD's tiles begin inside a group
    const double bytes = r * row_bytes * ((r * row_bytes < 4e6 ? 1.0 : rounds) + (astride ? 1 : 0)) + column * (share > r ? share / r : 1.0);
    if (bytes < best) best = bytes, rows = r;
  }
  const int last = mtiles % rows;
  return {FastDiv(mtiles * ntiles), FastDiv(rows * ntiles), FastDiv(rows), FastDiv(last ? last : rows), mtiles, mtiles * ntiles * ranges};
}

// The plan of a shape, remembered per thread: a serving loop asks for the same few again and again, from the host path and
// from the entry points.  `make` is a captureless lambda at one place in the source, so each has a table of its own.
template <typename Make>
auto cached_plan(int kind, int M, int N, int K, Make make) -> decltype(make(kind, M, N, K)) {
  struct Entry {
    int kind, M, N, K, cus;
    decltype(make(kind, M, N, K)) plan;
  };
  static thread_local Entry table[64] = {};
  const uint32_t h = ((uint32_t)M * 2654435761u ^ (uint32_t)N * 40503u ^ (uint32_t)K * 2246822519u ^ (uint32_t)kind) >> 7;
  Entry& e = table[h % 64];
  const int cus = device_cu_count();
  if (e.M != M || e.N != N || e.K != K || e.kind != kind || e.cus != cus) e = {kind, M, N, K, cus, make(kind, M, N, K)};
  return e.plan;
}

}  // namespace mi355q
