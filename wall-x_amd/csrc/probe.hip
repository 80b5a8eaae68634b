// Measurement probe: how fast one CU's MFMA pipes run bf16 instructions back to back on GIVEN operand values, with no
// LDS or memory traffic in the loop.  The rate depends on the values and on the order of the instructions (switching
// activity moves the sustained clock), so benchmarks time this on the same kind of data as the GEMM they are judging: in
// the GEMM kernels' own form it is the ceiling they can reach on that data, below the nominal peak.
//
// Benchmark-only: built into its own library (libwallx_probe.so) next to the product library, never linked into it
// and not part of its C ABI.
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace wx {
namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kProbeFrags = 8;       // operand fragments per wave, 16 bytes per lane each: four of A, then four of B
constexpr int kProbeMfmaPerIter = 32;

// FORM 0: 32x32x16, both operands change with every instruction.  1: 16x16x32, likewise.  2: 16x16x32 in the order of the
// GEMM kernels, where one operand changes.
template <int FORM>
__global__ __launch_bounds__(256, 1) void mfma_rate_kernel(const u32x4* __restrict__ operands, int iters,
                                                            float* __restrict__ sink) {
#if defined(__HIP_DEVICE_COMPILE__)
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  bf16x8 a[4], b[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    a[i] = __builtin_bit_cast(bf16x8, operands[(wave * kProbeFrags + i) * 64 + lane]);
    b[i] = __builtin_bit_cast(bf16x8, operands[(wave * kProbeFrags + 4 + i) * 64 + lane]);
  }
  float s = 0.f;
  if constexpr (FORM == 0) {
    f32x16 acc[4][2];  // 128 registers of independent accumulators
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) acc[i][j] = f32x16{};
    for (int it = 0; it < iters; ++it) {
#pragma unroll
      for (int u = 0; u < kProbeMfmaPerIter; ++u) {
        const int i = u % 4, j = (u + u / 4) % 4;
        acc[i][j % 2] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i], b[j], acc[i][j % 2], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);  // (in this order)
      }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) s += acc[i][0][r] + acc[i][1][r];
  } else {
    f32x4 acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{};
    for (int it = 0; it < iters; ++it) {
#pragma unroll
      for (int u = 0; u < kProbeMfmaPerIter; ++u) {
        const int i = FORM == 1 ? u % 4 : u / 4 % 4;
        const int j = FORM == 1 ? (u + u / 4) % 4 : (i & 1) ? 3 - u % 4 : u % 4;
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[j], a[i], acc[i][j], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) s += acc[i][j][r];
  }
  if (s == 123.456f) sink[0] = s;  // keeps the loop alive; practically never true
#endif
}

}  // namespace
}  // namespace wx

using namespace wx;

extern "C" size_t wxprobe_mfma_operand_bytes(void) { return static_cast<size_t>(4) * kProbeFrags * 64 * 16; }

// Runs `iters` x 32 MFMAs of `form` (above) per wave on every CU, operands (wxprobe_mfma_operand_bytes() bytes of bf16
// values, device memory, 16-byte aligned: [4 waves][4 fragments of A, 4 of B][64 lanes][8]) held in registers.
// *flops_per_launch (host pointer, may be NULL) receives the flops one launch performs; sink is one float of device memory
// that is practically never written.  Returns 0, -1 for bad arguments, -4 when the launch failed.
extern "C" int wxprobe_mfma_rate(const void* operands, int form, int iters, float* sink, double* flops_per_launch, void* stream) {
  if (!operands || !sink || (reinterpret_cast<uintptr_t>(operands) & 15) || form < 0 || form > 2 || iters < 1 || iters > (1 << 24))
    return -1;
  int dev = 0, cus = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0)
    return -4;
  if (flops_per_launch)
    *flops_per_launch = 2.0 * (form == 0 ? 32 * 32 * 16 : 16 * 16 * 32) * kProbeMfmaPerIter * static_cast<double>(iters) * 4 * cus;
  const auto kernel = form == 0 ? mfma_rate_kernel<0> : form == 1 ? mfma_rate_kernel<1> : mfma_rate_kernel<2>;
  hipLaunchKernelGGL(kernel, dim3(cus), dim3(256), 0, reinterpret_cast<hipStream_t>(stream),
                     static_cast<const u32x4*>(operands), iters, sink);
  return hipGetLastError() == hipSuccess ? 0 : -4;
}
