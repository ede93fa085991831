// Shared device helpers for the gfx950 kernels: element types, 64-lane wave reductions, error reporting.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdio.h>

#define JLLM_WAVE 64

// dtype codes shared with the Python side
enum { JLLM_F32 = 0, JLLM_BF16 = 1 };

struct bf16_t {
  uint16_t bits;
};

__device__ __forceinline__ float bf16_to_f32(bf16_t v) { return __uint_as_float(((uint32_t)v.bits) << 16); }

// round to nearest even; NaN stays NaN (quiet)
__device__ __forceinline__ bf16_t f32_to_bf16(float f) {
  uint32_t u = __float_as_uint(f);
  bf16_t r;
  if ((u & 0x7fffffffu) > 0x7f800000u) {
    r.bits = (uint16_t)((u >> 16) | 0x0040u);
    return r;
  }
  uint32_t lsb = (u >> 16) & 1u;
  u += 0x7fffu + lsb;
  r.bits = (uint16_t)(u >> 16);
  return r;
}

__device__ __forceinline__ float ldf(const float* p, size_t i) { return p[i]; }
__device__ __forceinline__ float ldf(const bf16_t* p, size_t i) { return bf16_to_f32(p[i]); }
// an entry of a bf16 or float32 vector as it lies in memory, for requests ahead of their use, and its value
__device__ __forceinline__ uint32_t raw_entry(const void* p, int dtype, int i) {
  return dtype == JLLM_BF16 ? (uint32_t)((const uint16_t*)p)[i] : ((const uint32_t*)p)[i];
}
__device__ __forceinline__ float raw_value(uint32_t raw, int dtype) { return __uint_as_float(dtype == JLLM_BF16 ? raw << 16 : raw); }
__device__ __forceinline__ void stf(float* p, size_t i, float v) { p[i] = v; }
__device__ __forceinline__ void stf(bf16_t* p, size_t i, float v) { p[i] = f32_to_bf16(v); }

// what a value becomes when it is stored in T and read back
template <typename T>
__device__ __forceinline__ float round_to(float v);
template <>
__device__ __forceinline__ float round_to<float>(float v) { return v; }
template <>
__device__ __forceinline__ float round_to<bf16_t>(float v) { return bf16_to_f32(f32_to_bf16(v)); }

// The gate function of the gated epilogue, out = gate(a . Wg, a . Wu), has a code that rides in bits 8 and up of an
// entry point's `epilogue` argument (bits 0..7: 0 store, 1 add into fp32, 2 gated), and one parameter, `gate_limit`,
// for the functions that have one. Built:
//   0 silu           z / (1 + exp(-z)) * u   (cpu/VectorKernels.java:637-639 of the reference)
//   1 gelu_tanh      0.5 z (1 + tanh(sqrt(2/pi) (z + 0.044715 z^3))) * u
//   2 swish_clamped  g = min(z, limit), v = clamp(u, -limit, limit): g / (1 + exp(-1.702 g)) * (v + 1)
// Every product kernel applies gated() below with the GateSpec its entry point made with JLLM_TAKE_GATE, which refuses a
// code that is not built with a message; another gate function is a case in gated(), a larger JLLM_GATE_COUNT, and a
// name in the Python face's table.
#define JLLM_GATE_SILU 0
#define JLLM_GATE_GELU_TANH 1
#define JLLM_GATE_SWISH_CLAMPED 2
#define JLLM_GATE_COUNT 3
#define JLLM_SWISH_ALPHA 1.702f
struct GateSpec {
  int fn;
  float limit;
};
#define JLLM_TAKE_GATE(name, epilogue, limit_, spec_)                                                        \
  GateSpec spec_;                                                                                            \
  do {                                                                                                       \
    const int gate_ = (epilogue) >> 8;                                                                       \
    (epilogue) &= 0xff;                                                                                      \
    if (gate_ < 0 || gate_ >= JLLM_GATE_COUNT)                                                               \
      JLLM_FAIL("%s: gate function %d of the gated epilogue is not built (0 silu, 1 gelu_tanh, 2 swish_clamped are)", name, gate_); \
    if (gate_ != 0 && (epilogue) != 2) JLLM_FAIL("%s: a gate function without the gated epilogue", name);    \
    if (gate_ == JLLM_GATE_SWISH_CLAMPED && !((limit_) > 0.f))                                               \
      JLLM_FAIL("%s: the clamped gate needs a positive limit, got %g", name, (double)(limit_));              \
    spec_.fn = gate_;                                                                                        \
    spec_.limit = (limit_);                                                                                  \
  } while (0)
// FAST: the hardware's exp2 and reciprocal (where the result is rounded to bf16 or added in fp32 anyway)
template <bool FAST>
__device__ __forceinline__ float sigmoid_times(float z, float slope) {  // z / (1 + exp(-slope z))
  if (FAST) return z * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-1.4426950408889634f * slope * z));
  return z / (1.0f + expf(-slope * z));
}
template <bool FAST>
__device__ __forceinline__ float gated(float z, float u, GateSpec gs) {
  if (gs.fn == JLLM_GATE_SILU) return sigmoid_times<FAST>(z, 1.0f) * u;
  if (gs.fn == JLLM_GATE_GELU_TANH) {
    const float inner = 0.7978845608028654f * (z + 0.044715f * z * z * z);
    if (FAST) return z * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-2.8853900817779268f * inner)) * u;  // 0.5 (1 + tanh x) = 1 / (1 + exp(-2x))
    return 0.5f * z * (1.0f + tanhf(inner)) * u;
  }
  const float g = fminf(z, gs.limit);
  const float v = fminf(fmaxf(u, -gs.limit), gs.limit);
  return sigmoid_times<FAST>(g, JLLM_SWISH_ALPHA) * (v + 1.0f);
}

// The scale of an RMSNorm from a row's sum of squares: the mean and the sum with eps in fp32, the inverse square root in
// double, rounded once to fp32 (cpu/VectorKernels.java:630-632 of the reference: (float)(1.0 / Math.sqrt(ss / n + eps))).
// The general kernels, which are the whole of a float32 run, use it; the bf16 matrix-core kernels keep an fp32 1/sqrt,
// which differs by at most one unit in the last place.
__device__ __forceinline__ float norm_scale(float ss, int n, float eps) {
  return (float)(1.0 / sqrt((double)(ss / (float)n + eps)));
}

// 2^(a - m), zero for a = -infinity whatever m is: the attention kernels keep scores in units of log2(e), so that the
// exponentials are single v_exp_f32 instructions
__device__ __forceinline__ float exp2_diff(float a, float m) { return a == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(a - m); }

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int o = JLLM_WAVE / 2; o > 0; o >>= 1) v += __shfl_xor(v, o, JLLM_WAVE);
  return v;
}

__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int o = JLLM_WAVE / 2; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, JLLM_WAVE));
  return v;
}

// Sum over a block of NW waves in a fixed order; every thread gets the result. `red` holds NW floats.
template <int NW>
__device__ __forceinline__ float block_sum(float v, float* red) {
  v = wave_sum(v);
  const int lane = threadIdx.x & (JLLM_WAVE - 1);
  const int w = threadIdx.x / JLLM_WAVE;
  __syncthreads();
  if (lane == 0) red[w] = v;
  __syncthreads();
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < NW; ++i) s += red[i];
  return s;
}

// Values that one workgroup leaves for another of the same launch. The compute units' caches, and the L2s of the eight dies,
// do not see each other's writes during a kernel; accesses of agent scope pass them by. So the data are stored and read with
// such accesses, a wave waits for its stores, and only then counts itself as arrived: who sees the count sees the data. (A
// fence of agent scope would write back and drop the whole L2 instead, which cost more than the launch it saves.) Nobody waits
// for anybody: the workgroup that arrives last does what is left to do.
__device__ __forceinline__ void store_shared2(float* p, float a, float b) {  // 8-byte aligned
  const unsigned long long v = (unsigned long long)__float_as_uint(a) | ((unsigned long long)__float_as_uint(b) << 32);
  __hip_atomic_store((unsigned long long*)p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void load_shared2(const float* p, float& a, float& b) {
  const unsigned long long v = __hip_atomic_load((const unsigned long long*)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  a = __uint_as_float((unsigned)v);
  b = __uint_as_float((unsigned)(v >> 32));
}
__device__ __forceinline__ void shared_stores_done() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }
// Called by one lane whose wave's (or, behind a barrier, whose workgroup's) stores are done: whether it is the last of `all`.
// The last one leaves the counter at zero for the next launch.
__device__ __forceinline__ bool arrived_last(int* counter, int all) {
  const int before = __hip_atomic_fetch_add(counter, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if (before != all - 1) return false;
  __hip_atomic_store(counter, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return true;
}

// host side -----------------------------------------------------------------------------------------------
void jllm_set_error(const char* fmt, ...);
extern "C" int jllm_compute_units();  // of the current GPU (elementwise.hip)
// sums fp32 partials [splits][M][N] in ascending order of the split, adds the bias, applies the epilogue (gemm_mfma.hip)
int jllm_splitk_reduce(const float* partial, int splits, const void* bias, int bias_dtype, void* out, int out_dtype,
                       int ldo, int M, int N, int epilogue, hipStream_t stream);

// the same for the accumulate epilogue, with the RMSNorm of the new rows (gemm_mfma.hip)
int jllm_splitk_reduce_norm(const float* partial, int splits, const void* bias, int bias_dtype, void* out, int out_dtype, int ldo, int M, int N,
                            int epilogue, const void* gain, int gain_dtype, float eps, void* rows, int ldr, hipStream_t stream);

#define JLLM_FAIL(...)           \
  do {                           \
    jllm_set_error(__VA_ARGS__); \
    return -1;                   \
  } while (0)

#define JLLM_CHECK_LAUNCH(name)                                               \
  do {                                                                        \
    hipError_t e_ = hipGetLastError();                                        \
    if (e_ != hipSuccess) JLLM_FAIL("%s: launch failed: %s", name, hipGetErrorString(e_)); \
  } while (0)

#define JLLM_DISPATCH_1(code, T, ...)                 \
  if ((code) == JLLM_F32) {                           \
    typedef float T;                                  \
    __VA_ARGS__                                       \
  } else if ((code) == JLLM_BF16) {                   \
    typedef bf16_t T;                                 \
    __VA_ARGS__                                       \
  } else {                                            \
    JLLM_FAIL("unknown dtype code %d", (int)(code));  \
  }
