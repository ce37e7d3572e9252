// Checks of the arithmetic that common.h and rows8.h state bit for bit, for the tests (in libmi355q_bench.so, not part of the product library): the short
// reciprocal, gate and division against the plain ones, over every operand they are stated for.
#include "../rows8.h"

using namespace mi355q;

namespace {

// Every float from 1 to 2^126
__global__ void __launch_bounds__(256) check_reciprocal_kernel(unsigned long long* wrong) {
  const uint32_t first = 0x3f800000u, last = 0x7e800000u;
  unsigned bad = 0;
  for (uint32_t v = first + blockIdx.x * 256 + threadIdx.x; v <= last; v += gridDim.x * 256) {
    const float s = bitcast<float>(v);
    bad += bitcast<uint32_t>(short_reciprocal(s)) != bitcast<uint32_t>(1.0f / s);
  }
  if (bad) atomicAdd(wrong, (unsigned long long)bad);
}

// Every gate with every up value: thread x's eight gates, 256 up values of a y.  (NaN: of any bits)
template <int DT>
__global__ void __launch_bounds__(256) check_gate_kernel(unsigned long long* wrong) {
  const uint32_t gate = (blockIdx.x * 256 + threadIdx.x) * 8;
  float a[8];
  for (int e = 0; e < 8; ++e) a[e] = Elem<DT>::to_f32((uint16_t)(gate + e));
  unsigned bad = 0;
  for (uint32_t up = blockIdx.y * 256; up < blockIdx.y * 256 + 256; ++up) {
    float b[8], y[8];
    for (int e = 0; e < 8; ++e) b[e] = Elem<DT>::to_f32((uint16_t)up);
    silu_mul8(a, b, y);
    for (int e = 0; e < 8; ++e) {
      const float want = Elem<DT>::to_f32(Elem<DT>::from_f32(silu_mul(a[e], b[e]))), got = Elem<DT>::to_f32(Elem<DT>::from_f32(y[e]));
      bad += bitcast<uint32_t>(got) != bitcast<uint32_t>(want) && !(got != got && want != want);
    }
  }
  if (bad) atomicAdd(wrong, (unsigned long long)bad);
}

// Every finite largest magnitude (one to a workgroup) with every value up to it, both signs: the codes of the per-token quantiser
template <int DT>
__global__ void __launch_bounds__(256) check_codes_kernel(unsigned long long* wrong) {
  const uint32_t top = blockIdx.x;                           // (positive 16-bit values are ordered as their bits)
  const float mx = Elem<DT>::to_f32((uint16_t)top), scale = fmaxf(mx, 1e-10f) / FP8_MAX;
  RowFp8 by(mx);
  unsigned bad = bitcast<uint32_t>(by.scale) != bitcast<uint32_t>(scale);
  for (uint32_t v = threadIdx.x * 4; v <= top; v += 256 * 4) {
    float y[8], want[8];
    for (int e = 0; e < 8; ++e) {
      const float x = Elem<DT>::to_f32((uint16_t)min(v + (e >> 1), top));
      y[e] = e & 1 ? -x : x;
      want[e] = clamp448(y[e] / scale);
    }
    const u2 codes = by.codes(y), wanted = to_fp8x8(want);
    bad += codes.x != wanted.x || codes.y != wanted.y;
  }
  if (bad) atomicAdd(wrong, (unsigned long long)bad);
}

}  // namespace

// what 0: reciprocals, 1: gates, 2: codes (1 and 2 for f16 or bf16).  Adds the number of differences to *wrong (device memory).  0 on success.
extern "C" int mi355q_bench_check_arithmetic(int what, int dtype, unsigned long long* wrong, void* stream) {
  if (!wrong || what < 0 || what > 2 || (dtype != MI355Q_F16 && dtype != MI355Q_BF16)) return 1;
  hipStream_t st = (hipStream_t)stream;
  const bool half = dtype == MI355Q_F16;
  if (what == 0) hipLaunchKernelGGL(check_reciprocal_kernel, dim3(4096), dim3(256), 0, st, wrong);
  else if (what == 1) hipLaunchKernelGGL(half ? check_gate_kernel<MI355Q_F16> : check_gate_kernel<MI355Q_BF16>, dim3(65536 / 8 / 256, 256), dim3(256), 0, st, wrong);
  else hipLaunchKernelGGL(half ? check_codes_kernel<MI355Q_F16> : check_codes_kernel<MI355Q_BF16>, dim3(half ? 0x7c00 : 0x7f80), dim3(256), 0, st, wrong);
  return hipGetLastError() == hipSuccess ? 0 : 2;
}
