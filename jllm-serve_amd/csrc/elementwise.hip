// Embedding gather, RMSNorm, and the error channel of the library.
#include <stdarg.h>
#include <string.h>

#include "common.h"
#include "layer_launches.h"

static thread_local char g_error[512] = "";

void jllm_set_error(const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_error, sizeof(g_error), fmt, ap);
  va_end(ap);
}

extern "C" const char* jllm_last_error() { return g_error; }

extern "C" int jllm_abi_version() { return 5; }

// Compute units of the current GPU, read from the device's properties once per device (0 on errors).
extern "C" int jllm_compute_units() {
  static int cached[64];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 0;
  if (cached[dev] == 0) {
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) return 0;
    cached[dev] = n;
  }
  return cached[dev];
}

// ---------------------------------------------------------------------------------------------------------
// x[t, :] = scale * E[ids[t], :]   (the residual stream is fp32 whatever the table's type)
template <typename T>
__global__ void embed_kernel(const T* __restrict__ table, const int* __restrict__ ids, float* __restrict__ out,
                             int d, float scale) {
  const int t = blockIdx.x;
  const size_t row = (size_t)ids[t] * d;
  float* o = out + (size_t)t * d;
  for (int i = threadIdx.x; i < d; i += blockDim.x) o[i] = ldf(table, row + i) * scale;
}

extern "C" int jllm_embed(const void* table, int table_dtype, const int* ids, float* out, int n_tokens, int d,
                          float scale, hipStream_t stream) {
  if (n_tokens <= 0) return 0;
  if (d <= 0) JLLM_FAIL("embed: width %d", d);
  JLLM_DISPATCH_1(table_dtype, T, {
    embed_kernel<T><<<n_tokens, 256, 0, stream>>>((const T*)table, ids, out, d, scale);
  })
  JLLM_CHECK_LAUNCH("embed");
  return 0;
}

// ---------------------------------------------------------------------------------------------------------
// RMSNorm of fp32 rows: y = (x * rsqrt(mean(x^2) + eps)) * g. One block per output row; `rows` (optional)
// picks the input row of each output row; output rows lie `ldo` elements apart. Sum of squares, the reciprocal root and both products are fp32.
// Rows of up to 8192 values whose width is a multiple of 4 are read once, 16 bytes per lane, and held in J vectors of registers
// per thread (J = 0: other widths take the two-pass loop); the loads are declared as aligned to an element only, which costs
// nothing, so that a row has the same bits wherever it and the gains lie. 2,048 rows of 4,096 13.4 -> 9.7 us (50 MB:
// 5.2 TB/s) since no branch stands around a load.
template <typename TG, typename TO, int J>
__global__ __launch_bounds__(256) void rmsnorm_kernel(const float* __restrict__ x, const int* __restrict__ rows,
                                                      const TG* __restrict__ gain, TO* __restrict__ out, int ldo, int d,
                                                      float eps) {
  __shared__ float red[4];
  const int r = blockIdx.x;
  const float* xi = x + (size_t)(rows ? rows[r] : r) * d;
  TO* o = out + (size_t)r * ldo;
  if constexpr (J > 0) {
    constexpr int JN = J > 0 ? J : 1;
    const int nv = d >> 2;
    float4 v[JN];
    TG gn[JN][4];
    int at[JN];
    float ss = 0.f;
    // the gains are requested together with the row; beyond the row's end its last four again (a branch around a load makes
    // the compiler wait for everything behind it)
#pragma unroll
    for (int j = 0; j < J; ++j) {
      at[j] = min((int)threadIdx.x + 256 * j, nv - 1);
      __builtin_memcpy(&v[j], xi + 4 * at[j], 16);
      __builtin_memcpy(gn[j], gain + 4 * at[j], 4 * sizeof(TG));
    }
#pragma unroll
    for (int j = 0; j < J; ++j)
      if ((int)threadIdx.x + 256 * j < nv) ss += v[j].x * v[j].x + v[j].y * v[j].y + v[j].z * v[j].z + v[j].w * v[j].w;
    ss = block_sum<4>(ss, red);
    const float s = norm_scale(ss, d, eps);
    const bool ovec = (((uintptr_t)o) & 15) == 0;
#pragma unroll
    for (int j = 0; j < J; ++j) {
      const int i = threadIdx.x + 256 * j;
      if (i < nv) {
        const float a = (v[j].x * s) * ldf(gn[j], 0), b = (v[j].y * s) * ldf(gn[j], 1), c = (v[j].z * s) * ldf(gn[j], 2), e = (v[j].w * s) * ldf(gn[j], 3);
        if (!ovec) {
          stf(o, 4 * i, a);
          stf(o, 4 * i + 1, b);
          stf(o, 4 * i + 2, c);
          stf(o, 4 * i + 3, e);
        } else if (sizeof(TO) == 2) {
          ((uint2*)o)[i] = uint2{(uint32_t)f32_to_bf16(a).bits | ((uint32_t)f32_to_bf16(b).bits << 16),
                                 (uint32_t)f32_to_bf16(c).bits | ((uint32_t)f32_to_bf16(e).bits << 16)};
        } else {
          ((float4*)o)[i] = float4{a, b, c, e};
        }
      }
    }
    return;
  }
  float ss = 0.f;
  for (int i = threadIdx.x; i < d; i += 256) {
    float v = xi[i];
    ss += v * v;
  }
  ss = block_sum<4>(ss, red);
  const float s = norm_scale(ss, d, eps);
  for (int i = threadIdx.x; i < d; i += 256) stf(o, i, (xi[i] * s) * ldf(gain, i));
}

extern "C" int jllm_rmsnorm(const float* x, const int* rows, int n_rows, int d, const void* gain, int gain_dtype,
                            float eps, void* out, int out_dtype, int ldo, hipStream_t stream) {
  if (n_rows <= 0) return 0;
  if (d <= 0) JLLM_FAIL("rmsnorm: width %d", d);
  if (ldo < d) JLLM_FAIL("rmsnorm: output row stride %d < width %d", ldo, d);
#define RN_CASE(J)                                                                                            \
  case J:                                                                                                      \
    rmsnorm_kernel<TG, TO, J><<<n_rows, 256, 0, stream>>>(x, rows, (const TG*)gain, (TO*)out, ldo, d, eps);     \
    break;
  JLLM_DISPATCH_1(gain_dtype, TG, {
    JLLM_DISPATCH_1(out_dtype, TO, {
      switch ((d & 3) == 0 && d <= 8192 ? (d / 4 + 255) / 256 : 0) {
        RN_CASE(0) RN_CASE(1) RN_CASE(2) RN_CASE(3) RN_CASE(4) RN_CASE(5) RN_CASE(6) RN_CASE(7) RN_CASE(8)
      }
    })
  })
#undef RN_CASE
  JLLM_CHECK_LAUNCH("rmsnorm");
  return 0;
}

// ---------------------------------------------------------------------------------------------------------
// Copies n 32-bit words. The source may be pinned host memory: the step's description (token ids, positions, block
// tables) reaches the device inside the stream of kernels, with no copy engine to start and wait for.
__global__ __launch_bounds__(256) void copy_words_kernel(const uint32_t* __restrict__ src, uint32_t* __restrict__ dst, size_t n) {
  const size_t n4 = n / 4;
  const size_t stride = (size_t)gridDim.x * 256;
  if ((((uintptr_t)src | (uintptr_t)dst) & 15) == 0) {
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n4; i += stride) ((uint4*)dst)[i] = ((const uint4*)src)[i];
    for (size_t i = n4 * 4 + (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += stride) dst[i] = src[i];
  } else {
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += stride) dst[i] = src[i];
  }
}

extern "C" int jllm_copy_words(const void* src, void* dst, long long n_words, hipStream_t stream) {
  if (n_words <= 0) return 0;
  if (((uintptr_t)src & 3) || ((uintptr_t)dst & 3)) JLLM_FAIL("copy_words: pointers must be 4-byte aligned");
  const long long groups = (n_words / 4 + 255) / 256;
  copy_words_kernel<<<(unsigned)(groups < 1 ? 1 : groups > 64 ? 64 : groups), 256, 0, stream>>>((const uint32_t*)src, (uint32_t*)dst,
                                                                                              (size_t)n_words);
  JLLM_CHECK_LAUNCH("copy_words");
  return 0;
}

// out[t] = [a[t] | b[t]] in out's type: two fp32 row sets (the stream and a second stream of the same width) side by
// side as the input rows of one product.
template <typename TO>
__global__ __launch_bounds__(256) void concat_rows_kernel(const float* __restrict__ a, const float* __restrict__ b, int d,
                                                         TO* __restrict__ out, int ldo) {
  const int t = blockIdx.x;
  for (int i = threadIdx.x; i < 2 * d; i += 256)
    stf(out + (size_t)t * ldo, i, i < d ? a[(size_t)t * d + i] : b[(size_t)t * d + i - d]);
}

extern "C" int jllm_concat_rows(const float* a, const float* b, int n_rows, int d, void* out, int out_dtype, int ldo,
                                hipStream_t stream) {
  if (n_rows <= 0) return 0;
  if (d <= 0 || ldo < 2 * d) JLLM_FAIL("concat_rows: rows of %d into rows of %d", d, ldo);
  JLLM_DISPATCH_1(out_dtype, TO, { concat_rows_kernel<TO><<<n_rows, 256, 0, stream>>>(a, b, d, (TO*)out, ldo); })
  JLLM_CHECK_LAUNCH("concat_rows");
  return 0;
}

// out[m][i] = src[m][rows[i]] of up to four matrices whose rows are lists of bytes: what goes on from a step's last layer, by one
// launch (a row list outside the matrix names its nearest row). A workgroup per row and matrix, in units of what every address and
// length of the matrix allows. Four rows of 4,096 bf16 and of 4,096 floats: 2.0 us inside a graph, two gathers of the library 5.4.
struct GatherRows {
  const unsigned char* src[4];
  unsigned char* out[4];
  long long ld[4], ldo[4], bytes[4];
};
template <typename U>
__device__ __forceinline__ void copy_row(const unsigned char* src, unsigned char* out, long long bytes) {
  for (long long i = threadIdx.x; i < bytes / (long long)sizeof(U); i += 256) ((U*)out)[i] = ((const U*)src)[i];
}
__global__ __launch_bounds__(256) void gather_rows_kernel(const int* __restrict__ rows, int n_from, GatherRows g) {
  const int m = blockIdx.y;
  const int from = min(max(rows[blockIdx.x], 0), n_from - 1);
  const unsigned char* src = g.src[m] + from * g.ld[m];
  unsigned char* out = g.out[m] + blockIdx.x * g.ldo[m];
  const uintptr_t all = (uintptr_t)g.src[m] | (uintptr_t)g.out[m] | (uintptr_t)g.ld[m] | (uintptr_t)g.ldo[m] | (uintptr_t)g.bytes[m];
  if ((all & 15) == 0)
    copy_row<uint4>(src, out, g.bytes[m]);
  else if ((all & 3) == 0)
    copy_row<uint32_t>(src, out, g.bytes[m]);
  else
    copy_row<uint16_t>(src, out, g.bytes[m]);
}

// `matrices`: of each the address of its first row and of the output's, the two row strides and a row's length, in bytes
extern "C" int jllm_gather_rows(const long long* matrices, int n_matrices, const int* rows, int n_rows, int n_from, hipStream_t stream) {
  if (n_rows <= 0) return 0;
  if (n_matrices < 1 || n_matrices > 4 || n_from <= 0) JLLM_FAIL("gather_rows: %d matrices (1 to 4) of %d rows", n_matrices, n_from);
  GatherRows g = {};
  for (int m = 0; m < n_matrices; ++m) {
    const long long* w = matrices + 5 * m;
    g.src[m] = (const unsigned char*)(uintptr_t)w[0], g.out[m] = (unsigned char*)(uintptr_t)w[1];
    g.ld[m] = w[2], g.ldo[m] = w[3], g.bytes[m] = w[4];
    if ((w[0] | w[1] | w[2] | w[3] | w[4]) & 1 || w[4] < 0 || w[2] < w[4] || w[3] < w[4])
      JLLM_FAIL("gather_rows: rows of %lld bytes, %lld apart, into rows %lld apart (even numbers, no rows that overlap)", w[4], w[2], w[3]);
  }
  gather_rows_kernel<<<dim3(n_rows, n_matrices), 256, 0, stream>>>(rows, n_from, g);
  JLLM_CHECK_LAUNCH("gather_rows");
  return 0;
}
