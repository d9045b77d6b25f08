// Measurement kernels (no counterpart in the reference): the read rate of the memory hierarchy, the engine clock
// during a run and the MFMA rate, the ceilings the optimizer's launches are compared against; and the MFMA layout check.
#include "common.h"

namespace psgdk {

// Each workgroup of 256 threads reads `iters` 4 KiB blocks of uint4: block (blockIdx * iters + i) * stride, its
// index wrapped into the buffer by `mask` (the buffer's uint4 count minus one, a power of two), so every load lies
// inside the buffer. stride 1 with grid * iters blocks = the buffer reads every byte once (HBM); an odd stride over a
// small buffer keeps it in the caches. The XOR of the loaded words is stored only when it equals a value that a
// buffer of one repeated byte never gives, so the loads stay and nothing is written.
__global__ void __launch_bounds__(256) read_rate_kernel(const uint4* __restrict__ buf, unsigned long long mask,
                                                        int iters, unsigned long long stride, unsigned* sink) {
  unsigned acc = 0;
#pragma unroll 8
  for (int i = 0; i < iters; ++i) {
    const unsigned long long blk = ((unsigned long long)blockIdx.x * (unsigned long long)iters + i) * stride;
    const uint4 v = buf[(blk * 256ull + threadIdx.x) & mask];
    acc ^= v.x ^ v.y ^ v.z ^ v.w;
  }
  if (acc == 0x9e3779b9u) sink[blockIdx.x] = acc;
}

hipError_t read_rate_launch(const void* buf, long long bytes, int wgs, int iters, long long stride, unsigned* sink,
                            hipStream_t st) {
  const unsigned long long mask = (unsigned long long)bytes / 16 - 1;
  hipLaunchKernelGGL(read_rate_kernel, dim3(wgs), dim3(256), 0, st, reinterpret_cast<const uint4*>(buf), mask, iters,
                     (unsigned long long)stride, sink);
  return hipGetLastError();
}

// One thread samples the engine clock: every step it sleeps (s_sleep 127, about 8 thousand cycles), then records
// the cycle counter and the constant-rate wall counter (out[2 i], out[2 i + 1]), for `samples` steps; the ratio of
// their increments times the wall counter's rate is the clock of the CU it runs on. Launched on a stream of its own
// beside the work being timed, it takes one wave of one CU.
__global__ void __launch_bounds__(64) clock_sample_kernel(int samples, unsigned long long* out) {
  if (threadIdx.x != 0) return;
  for (int i = 0; i < samples; ++i) {
    __builtin_amdgcn_s_sleep(127);
    out[2 * i] = (unsigned long long)clock64();
    out[2 * i + 1] = (unsigned long long)wall_clock64();
  }
}

// out[0] = the wall counter when the stream reaches this launch (marks a region for clock_sample_kernel's samples)
__global__ void __launch_bounds__(64) wall_mark_kernel(unsigned long long* out) {
  if (threadIdx.x == 0) out[0] = (unsigned long long)wall_clock64();
}

hipError_t clock_sample_launch(int samples, unsigned long long* out, hipStream_t st) {
  hipLaunchKernelGGL(clock_sample_kernel, dim3(1), dim3(64), 0, st, samples, out);
  return hipGetLastError();
}

hipError_t wall_mark_launch(unsigned long long* out, hipStream_t st) {
  hipLaunchKernelGGL(wall_mark_kernel, dim3(1), dim3(64), 0, st, out);
  return hipGetLastError();
}

// One MFMA on a single wave with operands placed by the lane layout the GEMM assumes; the host compares C with
// A @ B (layout check of the compiler builtins).
__global__ void psgdk_debug_mfma_kernel(const float* A, const float* B, float* C, int prec) {
  // A: 16 x K row-major, B: K x 16 row-major, C: 16 x 16, K = 32 (bf16) or 4 (fp32); one wave. prec 2: the 32 x 32
  // bf16 shape, A 32 x 16, B 16 x 32, C 32 x 32: lane l holds A[l % 32][8 (l / 32) + e] and B[8 (l / 32) + e][l % 32],
  // and accumulator m of lane l is C[8 (m / 4) + 4 (l / 32) + m % 4][l % 32].
  const int lane = threadIdx.x, r = lane & 15, g = lane >> 4;
  if (prec == 2) {
    const int c = lane & 31, h = lane >> 5;
    bf16x8_t a, b;
    for (int e = 0; e < 8; ++e) {
      a[e] = __builtin_bit_cast(__bf16, f32_to_bf16(A[c * 16 + 8 * h + e]));
      b[e] = __builtin_bit_cast(__bf16, f32_to_bf16(B[(8 * h + e) * 32 + c]));
    }
    f32x16_t acc;
    for (int m = 0; m < 16; ++m) acc[m] = 0.f;
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, acc, 0, 0, 0);
    for (int m = 0; m < 16; ++m) C[(8 * (m >> 2) + 4 * h + (m & 3)) * 32 + c] = acc[m];
    return;
  }
  f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
  if (prec == 1) {
    bf16x8_t a, b;
    for (int e = 0; e < 8; ++e) {
      a[e] = __builtin_bit_cast(__bf16, f32_to_bf16(A[r * 32 + g * 8 + e]));
      b[e] = __builtin_bit_cast(__bf16, f32_to_bf16(B[(g * 8 + e) * 16 + r]));
    }
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, acc, 0, 0, 0);
  } else {
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(A[r * 4 + g], B[g * 16 + r], acc, 0, 0, 0);
  }
  for (int e = 0; e < 4; ++e) C[(g * 4 + e) * 16 + r] = acc[e];
}

// The bf16 MFMA rate this GPU sustains at the moment of the call: each wave issues `iters` rounds of 32
// independent v_mfma_f32_16x16x32_bf16 (no memory traffic in the loop; operands from the lane index), and lane 0 of
// each wave writes the sum of its accumulators' first element to out[wave id] so that nothing is optimised away.
// 16384 flops per MFMA. One wave per SIMD issuing this instruction stays near 1.4-1.55 PFLOP/s however many
// independent accumulators it cycles through; two waves per SIMD with 32 each reach about 2.36 (measured): launch
// two workgroups per CU.
__global__ void __launch_bounds__(256, 2) psgdk_mfma_rate_kernel(int iters, float* out) {
  const int lane = threadIdx.x & 63;
  bf16x8_t a, b;
  for (int e = 0; e < 8; ++e) {
    a[e] = __builtin_bit_cast(__bf16, f32_to_bf16(1.f + 1e-3f * (lane + e)));
    b[e] = __builtin_bit_cast(__bf16, f32_to_bf16(1.f - 1e-3f * (lane ^ e)));
  }
  f32x4_t acc[32];
#pragma unroll
  for (int i = 0; i < 32; ++i) acc[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  for (int it = 0; it < iters; ++it) {
#pragma unroll
    for (int i = 0; i < 32; ++i) acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, acc[i], 0, 0, 0);
  }
  float t = 0.f;
#pragma unroll
  for (int i = 0; i < 32; ++i) t += acc[i][0];
  if (lane == 0) out[blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6)] = t;
}

hipError_t mfma_rate_launch(int iters, int wgs, float* out, hipStream_t st) {
  hipLaunchKernelGGL(psgdk_mfma_rate_kernel, dim3(wgs), dim3(256), 0, st, iters, out);
  return hipGetLastError();
}

hipError_t debug_mfma_launch(const float* A, const float* B, float* C, int prec, hipStream_t st) {
  hipLaunchKernelGGL(psgdk_debug_mfma_kernel, dim3(1), dim3(64), 0, st, A, B, C, prec);
  return hipGetLastError();
}

}  // namespace psgdk
