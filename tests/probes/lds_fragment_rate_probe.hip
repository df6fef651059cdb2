// Probe: the sustained full-chip rate of v_mfma_f32_32x32x16_bf16 whose one operand comes from LDS, as a function of how many
// products a 1 KB fragment read feeds (1, 2, 4). 256 workgroups of 8 waves, random bf16 operands, the reads one group of eight
// fragments ahead of their products; no global memory, barriers or vector work inside the loop. With one product per read LDS has to
// deliver 128 bytes a cycle, all it can; and every read costs power, which on a chip at its power limit is clock.
// Output: one line per number of products and repetition (the three alternate) with milliseconds and TFLOP/s.
// Built by tests/probes/build_probes.py, run by tests/test_probes_gpu.py; never part of the library.
#include <hip/hip_runtime.h>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <vector>
#define CK(x) do{hipError_t e=(x); if(e!=hipSuccess){printf("HIP error %s at %d\n", hipGetErrorString(e), __LINE__); exit(1);} }while(0)
typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(16))) float f32x16;

constexpr int kWaves = 8, kFrags = 8, kWaveElems = kFrags * 64 * 8;  // 8 KB of fragments per wave

// src: kWaves * kWaveElems values for LDS, then as many for the register operands
template <int N>
__global__ __launch_bounds__(kWaves * 64) void k_fragments(const __bf16* __restrict__ src, float* out, int iters) {
  __shared__ __attribute__((aligned(1024))) __bf16 smem[kWaves * kWaveElems];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const __bf16* const from = src + wave * kWaveElems + lane * 8;
  __bf16* const mine = smem + wave * kWaveElems;
  for (int f = 0; f < kFrags; ++f) *reinterpret_cast<bf16x8*>(mine + f * 512 + lane * 8) = *reinterpret_cast<const bf16x8*>(from + f * 512);
  bf16x8 b[4];
  for (int n = 0; n < 4; ++n) b[n] = *reinterpret_cast<const bf16x8*>(from + kWaves * kWaveElems + n * 512);
  __syncthreads();
  f32x16 acc[4] = {};
  bf16x8 a[kFrags];
  int at = lane * 8;
#pragma unroll
  for (int f = 0; f < kFrags; ++f) a[f] = *reinterpret_cast<const bf16x8*>(mine + f * 512 + at);
  for (int i = 0; i < iters; ++i) {
    asm volatile("" : "+v"(at));  // read again, not kept
#pragma unroll
    for (int f = 0; f < kFrags; ++f) {
      const bf16x8 now = a[f];
      a[f] = *reinterpret_cast<const bf16x8*>(mine + f * 512 + at);
#pragma unroll
      for (int n = 0; n < N; ++n) {
        const int j = (f * N + n) & 3;
        acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(now, b[n], acc[j], 0, 0, 0);
      }
    }
#pragma unroll
    for (int f = 0; f < kFrags; ++f) {
      __builtin_amdgcn_sched_group_barrier(0x008, N, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
  }
  float s = 0;
  for (int j = 0; j < 4; ++j)
    for (int v = 0; v < 16; ++v) s += acc[j][v];
  for (int f = 0; f < kFrags; ++f) s += (float)a[f][0];
  if (s == 1.2345f) out[0] = s;
}

static uint16_t f2bf(float f) { uint32_t u; memcpy(&u, &f, 4); u += 0x7fff + ((u >> 16) & 1); return u >> 16; }

int main() {
  std::vector<uint16_t> h(2 * kWaves * kWaveElems);
  srand(1);
  for (auto& x : h) {
    const float u1 = (rand() + 1.0f) / (RAND_MAX + 2.0f), u2 = (rand() + 1.0f) / (RAND_MAX + 2.0f);
    x = f2bf(sqrtf(-2 * logf(u1)) * cosf(6.2831853f * u2));
  }
  float* out;
  uint16_t* d;
  CK(hipMalloc(&out, 64));
  CK(hipMalloc(&d, h.size() * 2));
  CK(hipMemcpy(d, h.data(), h.size() * 2, hipMemcpyHostToDevice));
  hipEvent_t e0, e1;
  CK(hipEventCreate(&e0));
  CK(hipEventCreate(&e1));
  const int blocks = 256, products = 160000;  // per wave and launch
  auto launch = [&](int n) {
    const int iters = products / (kFrags * n);
    if (n == 1) hipLaunchKernelGGL(k_fragments<1>, dim3(blocks), dim3(kWaves * 64), 0, 0, (const __bf16*)d, out, iters);
    else if (n == 2) hipLaunchKernelGGL(k_fragments<2>, dim3(blocks), dim3(kWaves * 64), 0, 0, (const __bf16*)d, out, iters);
    else hipLaunchKernelGGL(k_fragments<4>, dim3(blocks), dim3(kWaves * 64), 0, 0, (const __bf16*)d, out, iters);
  };
  for (int rep = -1; rep < 5; ++rep)
    for (int n : {1, 2, 4}) {
      CK(hipEventRecord(e0));
      for (int i = 0; i < 3; ++i) launch(n);
      CK(hipEventRecord(e1));
      CK(hipEventSynchronize(e1));
      CK(hipGetLastError());
      float ms;
      CK(hipEventElapsedTime(&ms, e0, e1));
      ms /= 3;
      if (rep >= 0) printf("products per fragment read %d rep %d: %.3f ms  %.0f TFLOP/s\n", n, rep, ms, (double)blocks * kWaves * products * 32768.0 / ms * 1e-9);
      fflush(stdout);
    }
  return 0;
}
