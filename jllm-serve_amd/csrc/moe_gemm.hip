// The grouped products of a table-routed mixture of experts on the matrix cores, bf16 (the tiles, maps and epilogues
// of moe_generic.hip), for few rows per expert (decode steps): every needed expert's weights are streamed once per tile of
// up to 16 rows. (Steps that give the experts many rows each go through the grouped form of the tiled product,
// gemm_mfma.hip, which shares its operands through LDS.)
//
// What counts is how many bytes are on their way. A workgroup owns 32 weight rows of a tile's expert (16 outputs of the
// gated product: gate and up) and cuts K among its eight waves, 64 k (a whole 128-byte line of every row) at a time, so
// for K = 2,048 all of a wave's 16 KB of weights are requested at once; the waves' sums (MFMA 16x16x32, weight rows as the
// first operand, the tile's activation rows, gathered by the tile's row list, as the second) meet in LDS and are added in the
// order of the waves. With a wave per 64 outputs that walked K by itself, two steps ahead, gate/up of 20 experts of
// 1,024 x 2,048 took 50 us (3.3 TB/s) and down 26.
#include "common.h"
#include "mfma.h"

#define MM_WAVES 8
#define MM_K (MM_WAVES * 64)  // k per turn of the workgroup
#define MM_AHEAD 4            // turns whose loads are out together

template <bool GATED>
__global__ __launch_bounds__(MM_WAVES * 64, 4) void moe_gemm_mfma_kernel(
    const bf16_t* __restrict__ A, int lda, const bf16_t* __restrict__ W, const bf16_t* __restrict__ W2,
    void* __restrict__ out, int out_dtype, int ldo, int N, int K, const int* __restrict__ sorted,
    const int* __restrict__ tiles, int top, int in_map, int out_map, float weight, GateSpec gs) {
  __shared__ floatx4 red[MM_WAVES][2][64];
  const int tile = blockIdx.y;
  const int rows = tiles[3 * tile + 2];
  if (rows == 0) return;
  const int e = tiles[3 * tile], first = tiles[3 * tile + 1];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int sub = lane & 15, q4 = lane >> 4;
  const int n0 = blockIdx.x * (GATED ? 16 : 32);
  const int place = first + min(sub, rows - 1);
  const int asg = sorted[place];
  const bf16_t* xrow = A + (size_t)(in_map ? asg / top : place) * lda;
  // the two blocks of 16 weight rows: gate and up of the same outputs, or 32 neighbouring outputs (beyond N: the last row)
  const bf16_t* w0 = W + ((size_t)e * N + min(n0 + sub, N - 1)) * K;
  const bf16_t* w1 = GATED ? W2 + ((size_t)e * N + min(n0 + sub, N - 1)) * K : W + ((size_t)e * N + min(n0 + 16 + sub, N - 1)) * K;
  floatx4 acc0 = {0.f, 0.f, 0.f, 0.f}, acc1 = acc0;
  int k0 = wave * 64 + 8 * q4;  // this lane's first k; a turn holds two steps of 32
  for (; k0 - 8 * q4 + (MM_AHEAD - 1) * MM_K + 64 <= K; k0 += MM_AHEAD * MM_K) {
    u32x4 x[2 * MM_AHEAD], a[2 * MM_AHEAD], b[2 * MM_AHEAD];
#pragma unroll
    for (int i = 0; i < 2 * MM_AHEAD; ++i) {
      const int k = k0 + (i >> 1) * MM_K + (i & 1) * 32;
      a[i] = *(const u32x4*)(w0 + k);
      b[i] = *(const u32x4*)(w1 + k);
      x[i] = *(const u32x4*)(xrow + k);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < 2 * MM_AHEAD; ++i) {
      acc0 = mfma16(a[i], x[i], acc0);
      acc1 = mfma16(b[i], x[i], acc1);
    }
  }
  {  // what is left of the wave's K: places beyond the end are read inside the row and multiplied as zeros
    u32x4 x[2 * MM_AHEAD], a[2 * MM_AHEAD], b[2 * MM_AHEAD];
#pragma unroll
    for (int i = 0; i < 2 * MM_AHEAD; ++i) {
      const int k = k0 + (i >> 1) * MM_K + (i & 1) * 32;
      if (k - 8 * q4 >= K) continue;  // (the same in all lanes)
      const int at = k < K ? k : 0;
      a[i] = *(const u32x4*)(w0 + at);
      b[i] = *(const u32x4*)(w1 + at);
      x[i] = *(const u32x4*)(xrow + at);
    }
#pragma unroll
    for (int i = 0; i < 2 * MM_AHEAD; ++i) {
      const int k = k0 + (i >> 1) * MM_K + (i & 1) * 32;
      if (k - 8 * q4 >= K) continue;
      const u32x4 none = {0u, 0u, 0u, 0u};
      acc0 = mfma16(k < K ? a[i] : none, k < K ? x[i] : none, acc0);
      acc1 = mfma16(k < K ? b[i] : none, k < K ? x[i] : none, acc1);
    }
  }
  red[wave][0][lane] = acc0;
  red[wave][1][lane] = acc1;
  __syncthreads();
  if (wave >= (GATED ? 1 : 2)) return;
  floatx4 s0 = red[0][wave][lane], s1 = red[0][1][lane];
#pragma unroll
  for (int w = 1; w < MM_WAVES; ++w) {
    s0 += red[w][wave][lane];
    if (GATED) s1 += red[w][1][lane];
  }
  const int n = n0 + 16 * wave + 4 * q4;
  if (sub >= rows || n >= N) return;
  const size_t orow = out_map == 0 ? (size_t)place : out_map == 1 ? (size_t)asg : (size_t)(asg / top);
  float v[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = GATED ? gated<true>(s0[i], s1[i], gs) : s0[i];
  const size_t o = orow * ldo + n;
  if (out_map == 2) {
    floatx4* dst = (floatx4*)((float*)out + o);
    const floatx4 cur = *dst;
    *dst = floatx4{cur[0] + weight * v[0], cur[1] + weight * v[1], cur[2] + weight * v[2], cur[3] + weight * v[3]};
  } else if (out_dtype == JLLM_BF16) {
    *(u32x2*)((bf16_t*)out + o) = u32x2{pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3])};
  } else {
    *(floatx4*)((float*)out + o) = floatx4{v[0], v[1], v[2], v[3]};
  }
}

// returns 0 when it ran, 1 when the shape is not one it takes, -1 on errors
extern "C" int jllm_moe_gemm_bf16(const void* A, int a_dtype, int lda, const void* W, const void* W2, int w_dtype, void* out,
                                  int out_dtype, int ldo, int N, int K, const int* sorted, const int* tiles, int max_tiles,
                                  int tile_rows, int top, int in_map, int out_map, float weight, int epilogue,
                                  float gate_limit, hipStream_t stream) {
  if (max_tiles <= 0) return 0;
  if (a_dtype != JLLM_BF16 || w_dtype != JLLM_BF16) return 1;
  if (N <= 0 || K <= 0 || lda < K || ldo < N) JLLM_FAIL("moe_gemm: N %d K %d lda %d ldo %d", N, K, lda, ldo);
  if (tile_rows != 16) JLLM_FAIL("moe_gemm: this kernel takes tiles of 16 rows, the route made %d", tile_rows);
  JLLM_TAKE_GATE("moe_gemm", epilogue, gate_limit, gs);
  if ((epilogue != 0 && epilogue != 2) || (epilogue == 2) != (W2 != nullptr)) JLLM_FAIL("moe_gemm: epilogue %d", epilogue);
  if (in_map < 0 || in_map > 1 || out_map < 0 || out_map > 2) JLLM_FAIL("moe_gemm: maps %d / %d", in_map, out_map);
  if (out_map == 2 && (top != 1 || out_dtype != JLLM_F32)) JLLM_FAIL("moe_gemm: adding into the token's row needs top = 1 and fp32 rows");
  if (max_tiles > 65535) return 1;
  // 16-byte operand loads, 8- or 16-byte stores
  if ((K & 7) || (N & 3) || (lda & 7) || ((uintptr_t)A & 15) || ((uintptr_t)W & 15) || (W2 && ((uintptr_t)W2 & 15))) return 1;
  const int need = out_dtype == JLLM_BF16 ? 7 : 15;
  if (((uintptr_t)out & need) || (ldo & 3)) return 1;
  const int per_group = W2 ? 16 : 32;
  dim3 grid((N + per_group - 1) / per_group, max_tiles);
#define MM_LAUNCH(GATED)                                                                                                    \
  moe_gemm_mfma_kernel<GATED><<<grid, MM_WAVES * 64, 0, stream>>>((const bf16_t*)A, lda, (const bf16_t*)W, (const bf16_t*)W2, out, \
                                                                  out_dtype, ldo, N, K, sorted, tiles, top, in_map, out_map, weight, gs)
  if (W2)
    MM_LAUNCH(true);
  else
    MM_LAUNCH(false);
#undef MM_LAUNCH
  JLLM_CHECK_LAUNCH("moe_gemm_bf16");
  return 0;
}
