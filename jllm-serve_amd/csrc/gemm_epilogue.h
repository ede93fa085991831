// The epilogue of the tiled products: what a wave does with its accumulators once K is done.
//
// The weight fragment went in as the first MFMA operand, so an accumulator of 16 x 16 holds its tile transposed and a lane owns a run
// of four consecutive output columns of one row (lane l's at column (l / 16) * 4 of row l % 16), which it stores at once (in bf16 two
// neighbouring runs exchange halves between lanes first, so that a lane stores eight). `acc` holds a wave's runs, CN for each of its RM
// row blocks. Epilogues: store (fp32 or bf16), add into the
// fp32 residual, gated (runs [.][j] and [.][j + CN / 2] are gate and up of the same outputs: the gate function of
// common.h applied to both). With `split_z` the wave leaves an fp32 partial tile instead (K cut over workgroups; a
// reduction kernel applies bias and epilogue).
#pragma once
#include "common.h"
#include "mfma.h"

template <bool GATED, int RM, int CN, int TBM, int TBN>
__device__ __forceinline__ void tile_epilogue(floatx4 (&acc)[RM][CN], int lane, int wm, int wn, int m0, int n0,
                                              const void* __restrict__ bias, int bias_dtype, void* __restrict__ out,
                                              int out_dtype, int ldo, int M, int N, int epilogue, GateSpec gs, float* __restrict__ partial,
                                              int split_z, int n_splits) {
  constexpr int NI = GATED ? CN / 2 : CN;  // runs of outputs
  static_assert(NI % 2 == 0, "runs are stored in pairs");
  const int group = lane / 16;  // of lanes with the same columns
  const int row0 = m0 + wm * RM * 16 + lane % 16;
  const int col0 = n0 + wn * NI * 16 + group * 4;
  if (n_splits > 1) {  // partial sums [z][M][N]; the reduction kernel applies bias and epilogue
    float* pz = partial + (size_t)split_z * M * N;
#pragma unroll
    for (int mi = 0; mi < RM; ++mi) {
      const int m = row0 + mi * 16;
      if (m >= M) continue;
#pragma unroll
      for (int ni = 0; ni < CN; ++ni) {
        const int n = col0 + ni * 16;
        float* dst = pz + (size_t)m * N + n;
        if (n + 3 < N && (N & 3) == 0) {
          *(floatx4*)dst = acc[mi][ni];
        } else {
#pragma unroll
          for (int c = 0; c < 4; ++c)
            if (n + c < N) dst[c] = acc[mi][ni][c];
        }
      }
    }
    return;
  }
  const bool vec_ok = (ldo & 3) == 0 && (((uintptr_t)out) & 15) == 0;
  // Tiles that lie wholly inside the output (nearly all of a large product) take a path without per-element checks:
  // the kind of epilogue, the output type and the bias are decided once, outside the loops, and the gate's
  // 1 / (1 + exp(-x)) uses the hardware's exp2 and reciprocal (the result is rounded to bf16 or added in fp32 anyway).
  if (vec_ok && m0 + TBM <= M && n0 + (GATED ? TBN / 2 : TBN) <= N) {
    float bv[NI][4];
#pragma unroll
    for (int ni = 0; ni < NI; ++ni)
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const int n = col0 + ni * 16 + c;
        bv[ni][c] = !bias ? 0.f : (bias_dtype == JLLM_BF16) ? ldf((const bf16_t*)bias, n) : ldf((const float*)bias, n);
      }
    const int kind = epilogue == 1 ? 1 : out_dtype == JLLM_BF16 ? ((ldo & 7) == 0 ? 3 : 2) : 0;  // store fp32, add, store bf16 (in eights)
#pragma unroll
    for (int mi = 0; mi < RM; ++mi) {
      const size_t row = (size_t)(row0 + mi * 16) * ldo;
#pragma unroll
      for (int ni = 0; ni < NI; ni += 2) {
        floatx4 v[2];
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
          for (int c = 0; c < 4; ++c) {
            float x = acc[mi][ni + u][c] + bv[ni + u][c];
            if (GATED) x = gated<true>(x, acc[mi][GATED ? NI + ni + u : 0][c], gs);
            v[u][c] = x;
          }
        const size_t o = row + col0 + ni * 16;
        if (kind == 1) {
#pragma unroll
          for (int u = 0; u < 2; ++u) {
            floatx4* dst = (floatx4*)((float*)out + o + u * 16);
            const floatx4 cur = *dst;
            *dst = floatx4{cur[0] + v[u][0], cur[1] + v[u][1], cur[2] + v[u][2], cur[3] + v[u][3]};
          }
        } else if (kind == 0) {
#pragma unroll
          for (int u = 0; u < 2; ++u) *(floatx4*)((float*)out + o + u * 16) = v[u];
        } else {
          const u32x2 lo = {pack_bf16(v[0][0], v[0][1]), pack_bf16(v[0][2], v[0][3])};
          const u32x2 hi = {pack_bf16(v[1][0], v[1][1]), pack_bf16(v[1][2], v[1][3])};
          if (kind == 3) {
            // the odd lane groups' half of the first run against the even groups' half of the second: a lane then holds
            // eight neighbouring columns, of the first run's block in even groups, of the second's in odd ones
            const auto a = __builtin_amdgcn_permlane16_swap(lo.x, hi.x, false, false);
            const auto b = __builtin_amdgcn_permlane16_swap(lo.y, hi.y, false, false);
            *(u32x4*)((bf16_t*)out + o - group * 4 + (group & 1) * 16 + (group >> 1) * 8) = u32x4{a[0], b[0], a[1], b[1]};
          } else {
            *(u32x2*)((bf16_t*)out + o) = lo;
            *(u32x2*)((bf16_t*)out + o + 16) = hi;
          }
        }
      }
    }
    return;
  }
#pragma unroll
  for (int mi = 0; mi < RM; ++mi) {
    const int m = row0 + mi * 16;
    if (m >= M) continue;
#pragma unroll
    for (int ni = 0; ni < NI; ++ni) {
      const int n = col0 + ni * 16;
      if (n >= N) continue;
      float v[4];
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        float x = acc[mi][ni][c];
        if (bias && n + c < N) x += (bias_dtype == JLLM_BF16) ? ldf((const bf16_t*)bias, n + c) : ldf((const float*)bias, n + c);
        if (GATED) x = gated<true>(x, acc[mi][GATED ? NI + ni : 0][c], gs);
        v[c] = x;
      }
      const size_t o = (size_t)m * ldo + n;
      if (n + 3 < N && vec_ok) {
        if (epilogue == 1) {
          floatx4* dst = (floatx4*)((float*)out + o);
          floatx4 cur = *dst;
          *dst = floatx4{cur[0] + v[0], cur[1] + v[1], cur[2] + v[2], cur[3] + v[3]};
        } else if (out_dtype == JLLM_BF16) {
          *(u32x2*)((bf16_t*)out + o) = u32x2{pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3])};
        } else {
          *(floatx4*)((float*)out + o) = floatx4{v[0], v[1], v[2], v[3]};
        }
      } else {
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          if (n + c >= N) continue;
          if (epilogue == 1)
            ((float*)out)[o + c] += v[c];
          else if (out_dtype == JLLM_BF16)
            stf((bf16_t*)out, o + c, v[c]);
          else
            stf((float*)out, o + c, v[c]);
        }
      }
    }
  }
}
