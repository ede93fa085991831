// The grouped products of a table-routed mixture of experts on the matrix cores, bf16 (the tiles, maps and epilogues
// of moe_generic.hip), for few rows per expert (decode steps): every needed expert's weights are streamed once per tile of
// up to 16 rows. (Steps that give the experts many rows each go through the grouped form of the tiled product,
// gemm_mfma.hip, which shares its operands through LDS.)
//
// What counts is how many bytes are on their way. A workgroup owns 32 weight rows of a tile's expert (16 outputs of the
// gated product: gate and up) and cuts K among its eight waves, 256 k each in turn (four waves or two where K is no
// longer than theirs), so for K = 2,048 all of its weights are requested at once. The sums (MFMA 16x16x32, weight rows as the first
// operand, the tile's activation rows, gathered by the tile's row list, as the second) go from wave to wave through LDS:
// one accumulator per output takes its k in ascending order, as in the grouped form, so that a row's outputs have the same
// bits however many rows its experts get. Gate/up of 14 experts of 1,024 x 2,048 25 us, down 13; with a wave per 64
// outputs that walked K by itself, two steps ahead, 46 and 19; with a sum per wave, added at the end, 24 and 13 in other bits.
#include "common.h"
#include "mfma.h"

#define MM_STEPS 8  // steps of 32 k whose operands a wave holds

template <bool GATED, int WAVES>
__global__ __launch_bounds__(WAVES * 64, 4) void moe_gemm_mfma_kernel(
    const bf16_t* __restrict__ A, int lda, const bf16_t* __restrict__ W, const bf16_t* __restrict__ W2,
    void* __restrict__ out, int out_dtype, int ldo, int N, int K, const int* __restrict__ sorted,
    const int* __restrict__ tiles, int top, int in_map, int out_map, float weight, GateSpec gs) {
  constexpr int TURN = WAVES * MM_STEPS * 32;  // k per turn of the workgroup
  __shared__ floatx4 sums[2][64];
  __shared__ int asgs[16];  // the rows' assignments, for the stores (a register less while the operands are held)
  const int tile = blockIdx.y;
  const int rows = tiles[3 * tile + 2];
  if (rows == 0) return;
  const int e = tiles[3 * tile], first = tiles[3 * tile + 1];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int sub = lane & 15, q4 = lane >> 4;
  const int n0 = blockIdx.x * (GATED ? 16 : 32);
  const bf16_t* xrow;
  {
    const int place = first + min(sub, rows - 1), asg = sorted[place];
    if (threadIdx.x < 16) asgs[sub] = asg;
    xrow = A + (size_t)(in_map ? asg / top : place) * lda;
  }
  // the two blocks of 16 weight rows: gate and up of the same outputs, or 32 neighbouring outputs (beyond N: the last row)
  const bf16_t* w0 = W + ((size_t)e * N + min(n0 + sub, N - 1)) * K;
  const bf16_t* w1 = GATED ? W2 + ((size_t)e * N + min(n0 + sub, N - 1)) * K : W + ((size_t)e * N + min(n0 + 16 + sub, N - 1)) * K;
  u32x4 x[MM_STEPS], a[MM_STEPS], b[MM_STEPS];
  auto fetch = [&](int k0) {  // this wave's share of a turn; places beyond K are read at the row's start
    const bf16_t *p0 = w0 + k0 + 8 * q4, *p1 = w1 + k0 + 8 * q4, *px = xrow + k0 + 8 * q4;
    if (k0 + MM_STEPS * 32 <= K) {
#pragma unroll
      for (int i = 0; i < MM_STEPS; ++i) {
        a[i] = *(const u32x4*)(p0 + 32 * i);
        b[i] = *(const u32x4*)(p1 + 32 * i);
        x[i] = *(const u32x4*)(px + 32 * i);
      }
    } else {
#pragma unroll
      for (int i = 0; i < MM_STEPS; ++i) {
        const int by = k0 + 32 * i + 8 * q4 < K ? 32 * i : -(k0 + 8 * q4);
        a[i] = *(const u32x4*)(p0 + by);
        b[i] = *(const u32x4*)(p1 + by);
        x[i] = *(const u32x4*)(px + by);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  int k0 = wave * MM_STEPS * 32;
  if (k0 < K) fetch(k0);
  for (int turn = 0; turn < K; turn += TURN) {
    const int waves = min(WAVES, (K - turn + MM_STEPS * 32 - 1) / (MM_STEPS * 32));  // that have k in this turn
    for (int w = 0; w < waves; ++w) {
      if (w == wave) {
        floatx4 acc0 = {0.f, 0.f, 0.f, 0.f}, acc1 = acc0;
        if (k0 > 0) acc0 = sums[0][lane], acc1 = sums[1][lane];
        if (k0 + MM_STEPS * 32 <= K) {
#pragma unroll
          for (int i = 0; i < MM_STEPS; ++i) {
            acc0 = mfma16(a[i], x[i], acc0);
            acc1 = mfma16(b[i], x[i], acc1);
          }
        } else {  // the end of K: what was read beyond it counts as zeros
#pragma unroll
          for (int i = 0; i < MM_STEPS; ++i) {
            const bool in = k0 + 32 * i + 8 * q4 < K;
            const u32x4 none = {0u, 0u, 0u, 0u};
            acc0 = mfma16(in ? a[i] : none, in ? x[i] : none, acc0);
            acc1 = mfma16(in ? b[i] : none, in ? x[i] : none, acc1);
          }
        }
        sums[0][lane] = acc0;
        sums[1][lane] = acc1;
        k0 += TURN;
        if (k0 < K) fetch(k0);
      }
      __syncthreads();
    }
  }
  if (wave >= (GATED ? 1 : 2)) return;
  const floatx4 s0 = sums[wave][lane], s1 = sums[1][lane];
  const int n = n0 + 16 * wave + 4 * q4;
  if (sub >= rows || n >= N) return;
  const int place = first + sub, asg = asgs[sub];
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
#define MM_LAUNCH(GATED, WAVES)                                                                                             \
  moe_gemm_mfma_kernel<GATED, WAVES><<<grid, WAVES * 64, 0, stream>>>((const bf16_t*)A, lda, (const bf16_t*)W, (const bf16_t*)W2, out, \
                                                                      out_dtype, ldo, N, K, sorted, tiles, top, in_map, out_map, weight, gs)
#define MM_WAVES_OF(GATED)           \
  if (K <= 2 * MM_STEPS * 32)        \
    MM_LAUNCH(GATED, 2);             \
  else if (K <= 4 * MM_STEPS * 32)   \
    MM_LAUNCH(GATED, 4);             \
  else                               \
    MM_LAUNCH(GATED, 8);
  if (W2) {  // (no more waves than have k)
    MM_WAVES_OF(true)
  } else {
    MM_WAVES_OF(false)
  }
#undef MM_WAVES_OF
#undef MM_LAUNCH
  JLLM_CHECK_LAUNCH("moe_gemm_bf16");
  return 0;
}
