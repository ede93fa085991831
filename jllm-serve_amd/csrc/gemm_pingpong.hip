// out[M,N] = A[M,K] * W[N,K]^T for many rows, bf16 on the matrix cores (v_mfma_f32_16x16x32_bf16).
//
//  * A workgroup of 8 waves (2 x 4; 1 x 8 for the wide tiles further down) owns a 256 x 256 output tile (a wave 128 x 64: 8 by
//    4 accumulators of 16 x 16). (The 16 x 16 x 32 form rather than 32 x 32 x 16: the full chip is bound by its power, and
//    a multiply-add of the smaller form reads and writes half as many accumulator bytes.)
//  * K advances in stages of 64, so that a load covers whole lines of 128 bytes, eight rows to an instruction. A stage is four
//    units of LDS: each operand's first half (for every wave the first half of its rows, of its columns) and second. Two
//    units are a pair, which is what the ring in LDS holds: even pairs the first halves A0 and B0 of a stage, odd ones its
//    B1 and A1. Five pairs of 32 KB are all of the 160 KB.
//  * Global -> LDS without registers (global_load_lds_dwordx4), three to four pairs ahead. A lane's place in LDS is fixed by its
//    number, so the bank swizzle is applied on the global side (ring_swz).
//  * A wave multiplies half a stage between two barriers, A0 with B0 and B1, then A1 with both: 32 MFMAs, whose operands are
//    all in registers when the half begins except for B1, and between them, evenly, the 12 LDS reads of the next pair and its 4 loads.
//    Nothing is a phase of its own: of the two waves of a SIMD whichever is free multiplies, and the pipe of the
//    loads, which fills a compute unit's LDS at 32 bytes a clock and would be busy all the time at the matrix cores' full rate, is
//    asked evenly. A half takes 1,172 clocks of the 1,024 that its MFMAs alone take; what is left is the clock, which the
//    chip's power holds at 1.6 to 1.75 GHz (MFMAs on operands that do not change run at 2.37).
//
// What stood here before (stages of 32, the waves in two groups half a stage apart, one multiplying while the other read LDS
// and loaded, a barrier after every phase) / this, us, plain loops over changing weights: 8B gate/up at 2,048 rows 328 / 287 (1.44
// PFLOP/s; the library's plain product of that size 275), qkv 96 / 84, down in two parts 178 / 145, 14B gate/up at 4,608
// rows 1,488 / 1,150 (the library 1,323). No difference: the order of the multiplies inside a half, the loads early or late
// in it, priorities. Four waves of 128 x 128 (a third fewer LDS reads, a 5 % higher clock, 1,215 clocks a half): 3 % slower.
//
// Order of the tiles: a die (every eighth workgroup) takes a run of neighbouring tiles, in bands of four columns and row by row
// inside a band, so that its 32 workgroups work on about eight by four tiles and its L2 passes on fewer operands (what they cost
// is power, too): 14B gate/up at 4,608 rows 1,333 -> 1,188 us, 8B down 158 -> 149, gate/up at 2,048 rows 301 -> 297; without the loads' even spread
// it made no difference.
//
// A second tile has 192 rows (a wave 96 x 64): it moves a sixth more bytes per multiply, but where it fills the rounds of
// workgroups better it is ahead (900 rows of the 8B shape's gate/up are 480 tiles in two rounds instead of 384 in two).
//
// Epilogues as in the other tiled kernel (gemm_epilogue.h). Needs K % 32 == 0 (of a last stage of 32 only the first half is
// multiplied) and K >= 128, 16-byte aligned rows; any M and N (rows beyond the end are read as the last row and never stored).
#include <type_traits>
#include "common.h"
#include "layer_launches.h"
#include "lds_ring.h"
#include "gemm_epilogue.h"
#include "mfma.h"

#define PP_BK 64
#define PP_ROW_BYTES (PP_BK * 2)  // a tile row in LDS: 128 bytes = 8 pieces of 16
#define PP_WAVES 8
#define PP_FENCE() __builtin_amdgcn_sched_barrier(0)

// the ring of a tile of 32 FM rows for each of WGM waves and 64 columns for each of 8 / WGM
template <int FM, int WGM>
struct PingpongRing {
  static constexpr int WGN = PP_WAVES / WGM;
  static constexpr int A_UNIT = WGM * FM * 16 * PP_ROW_BYTES, B_UNIT = WGN * 32 * PP_ROW_BYTES, PAIR = A_UNIT + B_UNIT;
  static constexpr int PAIRS = 160 * 1024 / PAIR < 5 ? 160 * 1024 / PAIR : 5, BYTES = PAIRS * PAIR;
  static_assert(PAIRS >= 4, "one being read, one that must have landed, one on its way, one that others may still read");
};

// WGM x 8 / WGM waves of 32 FM rows by 64 columns each: the tile whose first row and first output are m0 and n0
template <bool GATED, int FM, int WGM>
__device__ __forceinline__ void pingpong_tile(
    const bf16_t* __restrict__ A, int lda, const bf16_t* __restrict__ W, const bf16_t* __restrict__ W2,
    const void* __restrict__ bias, int bias_dtype, void* __restrict__ out, int out_dtype, int ldo, int M, int N, int K,
    int epilogue, GateSpec gs, float* __restrict__ partial, int m0, int n0) {
  using Ring = PingpongRing<FM, WGM>;
  constexpr int WGN = Ring::WGN, NP = Ring::PAIRS, PAIR = Ring::PAIR;
  constexpr int TBM = WGM * FM * 32, TBN = WGN * 64;
  // load instructions (8 rows each) per wave and unit. Where A's unit is 12 or 4 of them, the first four waves take one more.
  constexpr int NA = WGM * FM * 2, LA = (NA + PP_WAVES - 1) / PP_WAVES, LA1 = NA * 2 / PP_WAVES - LA, LB = WGN * 4 / PP_WAVES;
  static_assert((LA + LA1) * PP_WAVES / 2 == NA && LA - LA1 <= 1, "the first four waves take LA, the others LA1");
  constexpr int L0 = LA + LB, L1 = LA1 + LB;
  constexpr int NM = 8 * FM, AHEAD = NP - 3;  // multiplies of half a stage; pairs that may be on their way at its end
  extern __shared__ __align__(1024) unsigned char smem[];
  const int tid = threadIdx.x;
  // the wave's number is the same in all its lanes: said so, its part of the tile and the places in LDS it fills stay in
  // scalar registers
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const bool first = wave < PP_WAVES / 2;
  const int wm = wave / WGN, wn = wave % WGN;
  const int nk_all = (K + PP_BK - 1) / PP_BK;
  const int nk_per = (nk_all + gridDim.z - 1) / gridDim.z;
  const int kt0 = blockIdx.z * nk_per;
  const int nk = max(0, min(nk_all, kt0 + nk_per) - kt0), pairs = 2 * nk;
  const bool half_k = (K & 32) != 0;  // the last stage of K is 32 long

  // ---- global side of the loads: an operand's start at this workgroup's first stage (the same in all lanes, advanced by scalar
  // arithmetic) plus a 32-bit byte offset per lane that never changes (row and piece; rows x row length < 4 GB: checked on the host)
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)smem;
  const unsigned char* abase = (const unsigned char*)A + (size_t)kt0 * PP_ROW_BYTES;
  const unsigned char* wbase[2] = {(const unsigned char*)W + (size_t)kt0 * PP_ROW_BYTES,
                                   (const unsigned char*)(GATED ? W2 : W) + (size_t)kt0 * PP_ROW_BYTES};
  uint32_t aoff[2][LA], boff[2][LB];
  const int achunk = LA == LA1 || first ? wave * LA : PP_WAVES / 2 * LA + (wave - PP_WAVES / 2) * LA1;  // (the others' c = LA1 is never asked for)
#pragma unroll
  for (int u = 0; u < 2; ++u) {
#pragma unroll
    for (int c = 0; c < LA; ++c) {
      const int r = (achunk + c) * 8 + (lane >> 3);  // row r of the unit: row r % 16 FM of the half of wave row r / 16 FM
      const int row = r / (FM * 16) * (FM * 32) + u * FM * 16 + r % (FM * 16);
      aoff[u][c] = (uint32_t)min(m0 + row, M - 1) * (uint32_t)lda * 2u + (uint32_t)(((lane & 7) ^ ring_swz(r)) * 16);
    }
#pragma unroll
    for (int c = 0; c < LB; ++c) {
      const int r = (wave * LB + c) * 8 + (lane >> 3);  // gated: B0 is the gate's rows, B1 the up weight's of the same outputs
      const int row = GATED ? n0 + r : n0 + (r >> 5) * 64 + u * 32 + (r & 31);
      boff[u][c] = (uint32_t)min(row, N - 1) * (uint32_t)K * 2u + (uint32_t)(((lane & 7) ^ ring_swz(r)) * 16);
    }
  }
  const uint32_t adst = lds0 + achunk * 8 * PP_ROW_BYTES, bdst = lds0 + Ring::A_UNIT + wave * LB * 8 * PP_ROW_BYTES;
  // Load l of pair p into the slot at byte `slot`. Of a last stage of 32 the lanes of its second half read the first again, which
  // is never multiplied; `whole`: not that stage. (Bit 2 of a lane's piece is that of lane ^ lane / 8, whatever the row.)
  const uint32_t second = (uint32_t)((lane ^ (lane >> 3)) & 4) * 16;
  auto load = [&](int p, uint32_t slot, int l, bool whole) {
    const size_t kbytes = (size_t)(p >> 1) * PP_ROW_BYTES;
    const uint32_t back = !whole && half_k && kt0 + (p >> 1) == nk_all - 1 ? second : 0u;
    if (l < LA) {
      if (l >= LA1 && !first) return;
      load_to_lds_16(abase + kbytes, aoff[p & 1][l] - back, adst + slot + l * 1024);
    } else {
      load_to_lds_16(wbase[p & 1] + kbytes, boff[p & 1][l - LA] - back, bdst + slot + (l - LA) * 1024);
    }
  };
  auto landed = [&](int left) {  // until at most `left` pairs of the wave's loads are on their way
    if (LA == LA1 || first) {
      if (AHEAD >= 2 && left >= 2) wait_loads<2 * L0>();
      else if (left >= 1) wait_loads<L0>();
      else wait_loads<0>();
    } else {
      if (AHEAD >= 2 && left >= 2) wait_loads<2 * L1>();
      else if (left >= 1) wait_loads<L1>();
      else wait_loads<0>();
    }
  };

  // ---- LDS side: fragment of a block of 16 rows: row = block * 16 + lane % 16, piece = lane / 16 (16 bytes: 8 of 32 k), + 4 for the
  // stage's second 32 (bit 6 of the address); 16 rows further leaves ring_swz unchanged
  const int ra = wm * FM * 16 + (lane & 15), rb = wn * 32 + (lane & 15);
  const int aread = ra * PP_ROW_BYTES + (((lane >> 4) ^ ring_swz(ra)) * 16);
  const int bread = Ring::A_UNIT + rb * PP_ROW_BYTES + (((lane >> 4) ^ ring_swz(rb)) * 16);
  u32x4 fa[2][2][FM], fb[2][2][2];  // [half of the rows, of the columns][32 of k][block]
  auto read_a = [&](int u, uint32_t slot, int x) {
    fa[u][x / FM][x % FM] = *(const u32x4*)(smem + slot + (aread ^ (x / FM * 64)) + x % FM * 16 * PP_ROW_BYTES);
  };
  auto read_b = [&](int u, uint32_t slot, int x) {
    fb[u][x / 2][x % 2] = *(const u32x4*)(smem + slot + (bread ^ (x / 2 * 64)) + x % 2 * 16 * PP_ROW_BYTES);
  };
  floatx4 acc[2 * FM][4];
#pragma unroll
  for (int i = 0; i < 2 * FM; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};

  // ---- prologue: all pairs but one on their way, the first two landed, the first in registers
#pragma unroll
  for (int p = 0; p < NP - 1; ++p)
    if (p < pairs) {
#pragma unroll
      for (int l = 0; l < L0; ++l) load(p, p * PAIR, l, false);
    }
  landed(pairs >= NP - 1 ? AHEAD : 0);
  PP_FENCE();
  __builtin_amdgcn_s_barrier();
  PP_FENCE();
#pragma unroll
  for (int x = 0; x < 2 * FM; ++x) read_a(0, 0, x);
#pragma unroll
  for (int x = 0; x < 4; ++x) read_b(0, 0, x);
  // Half h of the whole product reads pair h + 1 (its slot: rs) and loads pair h + NP - 1 into the slot of pair h - 1 (ws), which
  // every wave had in registers, and multiplied, before the barrier behind half h - 1. At its end pair h + 2 has landed: each wave waits for
  // its own loads, the barrier for all waves.
  uint32_t rs = PAIR, ws = (NP - 1) * PAIR;
  auto half = [&](auto which, auto full, int t) {
    constexpr int H = decltype(which)::value;
    constexpr bool FULL = decltype(full)::value;  // not among the last stages: every load is asked for
    const int p = 2 * t + H + NP - 1;
#pragma unroll
    for (int n = 0; n < NM; ++n) {
      const int q = n / (NM / 2), kk = n / (NM / 4) % 2, i = n % (NM / 4) / 2, j = n % 2;
      if (FULL || !(kk && half_k && kt0 + t == nk_all - 1)) acc[H * FM + i][q * 2 + j] = mfma16(fb[q][kk][j], fa[H][kk][i], acc[H * FM + i][q * 2 + j]);
      PP_FENCE();
      // B1 is read first, used a quarter later; A0 of the next stage while A1 is multiplied, its B0 behind the last use of this one's
      if (n % 2 == 0) {
        const int x = n / 2;
        if (H == 0) {
          if (x < 4) read_b(1, rs, x);
          else if (x < 4 + 2 * FM) read_a(1, rs, x - 4);
        } else {
          if (x < 2 * FM) read_a(0, rs, x);
          else if (x < 2 * FM + 4) read_b(0, rs, x - 2 * FM);
        }
        PP_FENCE();
      }
      constexpr int EVERY = NM / L0;
      if (n % EVERY == EVERY / 2 && n / EVERY < L0 && (FULL || p < pairs)) {
        load(p, ws, n / EVERY, FULL);
        PP_FENCE();
      }
    }
    landed(FULL ? AHEAD : min(p, pairs - 1) - (2 * t + H + 2));
    PP_FENCE();
    __builtin_amdgcn_s_barrier();
    PP_FENCE();
    rs = rs == (NP - 1) * PAIR ? 0 : rs + PAIR;
    ws = ws == (NP - 1) * PAIR ? 0 : ws + PAIR;
  };
  int t = 0;
  for (; t < nk - (half_k ? 3 : 2); ++t) {
    half(std::integral_constant<int, 0>{}, std::true_type{}, t);
    half(std::integral_constant<int, 1>{}, std::true_type{}, t);
  }
  for (; t < nk; ++t) {  // (the reads behind the last stage fetch some slot's bytes, which are never multiplied)
    half(std::integral_constant<int, 0>{}, std::false_type{}, t);
    half(std::integral_constant<int, 1>{}, std::false_type{}, t);
  }
  tile_epilogue<GATED, 2 * FM, 4, TBM, TBN>(acc, lane, wm, wn, m0, n0, bias, bias_dtype, out, out_dtype, ldo, M, N, epilogue, gs, partial,
                                                (int)blockIdx.z, (int)gridDim.z);
}

// Which tile workgroup b of rows x cols takes: workgroups b, b + 8, b + 16 .. share a die, which gets a run of neighbouring tiles,
// in bands of four columns, row by row inside a band
__device__ __forceinline__ void die_tile(int b, int rows, int cols, int& row, int& col) {
  const int tiles = rows * cols, each = tiles >> 3, more = tiles & 7, die = b & 7;
  const int i = die * each + min(die, more) + (b >> 3);
  const int band = i / (4 * rows), r = i - band * 4 * rows, width = min(4, cols - band * 4);
  row = r / width;
  col = band * 4 + r - row * width;
}

template <bool GATED, int FM>
__global__ __launch_bounds__(PP_WAVES * 64) void gemm_pingpong_kernel(
    const bf16_t* __restrict__ A, int lda, const bf16_t* __restrict__ W, const bf16_t* __restrict__ W2,
    const void* __restrict__ bias, int bias_dtype, void* __restrict__ out, int out_dtype, int ldo, int M, int N, int K,
    int epilogue, GateSpec gs, float* __restrict__ partial) {
  int row, col;
  die_tile(blockIdx.x + blockIdx.y * gridDim.x, gridDim.y, gridDim.x, row, col);
  pingpong_tile<GATED, FM, 2>(A, lda, W, W2, bias, bias_dtype, out, out_dtype, ldo, M, N, K, epilogue, gs, partial, row * 64 * FM, col * (GATED ? 128 : 256));
}

// Tiles of 256 x 256 and, for the last rows where those are at most 128, of 128 x 512 (64 x 512 where they are at most 64): `wide`
// of the latter, which come first because they take longer, then rows of `cols` of the former. A tile of 256 rows of which a few
// are there takes as long as a full one, and so does the round of workgroups that it begins. A wide tile takes half as many
// workgroups; its stage moves a quarter (an eighth) more bytes into LDS and takes 1.13 (1.03) times as long. us, the best of whole tiles of
// any size / this: gate/up of the 8B shape at 560 rows (288 tiles / 240) 125.7 / 98.7, at 631 131.4 / 104.4, of the 14B shape at 300 182.7 / 138.9,
// at 1,320 392.8 / 370.4, at 4,614 (10.1 rounds / 9.8) 1,285 / 1,189, of the 32B shape at 600 351.6 / 305.9; 14B down at 3,111 484.1 / 406.8, 4B
// qkv at 2,600 79.8 / 64.9. Last rows of 129 to 192 in a tile of either kind gained nothing.
template <bool GATED>
__global__ __launch_bounds__(PP_WAVES * 64) void gemm_pingpong_mixed_kernel(
    const bf16_t* __restrict__ A, int lda, const bf16_t* __restrict__ W, const bf16_t* __restrict__ W2,
    const void* __restrict__ bias, int bias_dtype, void* __restrict__ out, int out_dtype, int ldo, int M, int N, int K,
    int epilogue, GateSpec gs, float* __restrict__ partial, int wide, int cols) {
  const int whole = M >> 8 << 8, b = blockIdx.x;
  if (b >= wide) {
    int row, col;
    die_tile(b - wide, M >> 8, cols, row, col);
    pingpong_tile<GATED, 4, 2>(A, lda, W, W2, bias, bias_dtype, out, out_dtype, ldo, M, N, K, epilogue, gs, partial, row * 256, col * (GATED ? 128 : 256));
  } else if (M - whole > 64) {
    pingpong_tile<GATED, 4, 1>(A, lda, W, W2, bias, bias_dtype, out, out_dtype, ldo, M, N, K, epilogue, gs, partial, whole, b * (GATED ? 256 : 512));
  } else {
    pingpong_tile<GATED, 2, 1>(A, lda, W, W2, bias, bias_dtype, out, out_dtype, ldo, M, N, K, epilogue, gs, partial, whole, b * (GATED ? 256 : 512));
  }
}

template <int FM>
static int launch_pingpong(const void* A, int lda, const void* W, const void* W2, const void* bias, int bias_dtype,
                           void* out, int out_dtype, int ldo, int M, int N, int K, int epilogue, GateSpec gs, int splits,
                           float* partial, hipStream_t stream) {
  constexpr int TBM = 4 * FM * 16, TBN = 256;
  const int cols = W2 ? TBN / 2 : TBN;
  dim3 grid((N + cols - 1) / cols, (M + TBM - 1) / TBM, splits);
  if (grid.y > 65535) return 1;
  constexpr size_t smem = PingpongRing<FM, 2>::BYTES;
  static bool configured = false;
  if (!configured) {
    hipError_t e1 = hipFuncSetAttribute((const void*)gemm_pingpong_kernel<true, FM>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
    hipError_t e2 = hipFuncSetAttribute((const void*)gemm_pingpong_kernel<false, FM>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
    if (e1 != hipSuccess || e2 != hipSuccess) JLLM_FAIL("gemm_pingpong: cannot reserve %zu bytes of LDS", smem);
    configured = true;
  }
  if (W2)
    gemm_pingpong_kernel<true, FM><<<grid, PP_WAVES * 64, smem, stream>>>(
        (const bf16_t*)A, lda, (const bf16_t*)W, (const bf16_t*)W2, bias, bias_dtype, out, out_dtype, ldo, M, N, K, epilogue, gs, partial);
  else
    gemm_pingpong_kernel<false, FM><<<grid, PP_WAVES * 64, smem, stream>>>(
        (const bf16_t*)A, lda, (const bf16_t*)W, nullptr, bias, bias_dtype, out, out_dtype, ldo, M, N, K, epilogue, gs, partial);
  return 0;
}

static int launch_mixed(const void* A, int lda, const void* W, const void* W2, const void* bias, int bias_dtype,
                        void* out, int out_dtype, int ldo, int M, int N, int K, int epilogue, GateSpec gs, int splits,
                        float* partial, hipStream_t stream) {
  const int cols = (N + (W2 ? 127 : 255)) / (W2 ? 128 : 256), wide = (cols + 1) / 2;
  const long groups = (long)(M / 256) * cols + wide;
  if (groups > 0x7fffffffl) return 1;
  constexpr size_t smem = 160 * 1024;  // of the largest of the three rings
  static_assert(PingpongRing<4, 2>::BYTES <= smem && PingpongRing<4, 1>::BYTES <= smem && PingpongRing<2, 1>::BYTES <= smem, "all fit");
  static bool configured = false;
  if (!configured) {
    hipError_t e1 = hipFuncSetAttribute((const void*)gemm_pingpong_mixed_kernel<true>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
    hipError_t e2 = hipFuncSetAttribute((const void*)gemm_pingpong_mixed_kernel<false>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
    if (e1 != hipSuccess || e2 != hipSuccess) JLLM_FAIL("gemm_pingpong: cannot reserve %zu bytes of LDS", smem);
    configured = true;
  }
  dim3 grid((unsigned)groups, 1, splits);
  if (W2)
    gemm_pingpong_mixed_kernel<true><<<grid, PP_WAVES * 64, smem, stream>>>(
        (const bf16_t*)A, lda, (const bf16_t*)W, (const bf16_t*)W2, bias, bias_dtype, out, out_dtype, ldo, M, N, K, epilogue, gs, partial, wide, cols);
  else
    gemm_pingpong_mixed_kernel<false><<<grid, PP_WAVES * 64, smem, stream>>>(
        (const bf16_t*)A, lda, (const bf16_t*)W, nullptr, bias, bias_dtype, out, out_dtype, ldo, M, N, K, epilogue, gs, partial, wide, cols);
  return 0;
}

// `tile_rows`: 256 or 192 (rows of the output tile; 256 columns, 128 outputs with the gated epilogue), or 384: tiles of 256 rows and
// wide ones for the last at most 128 rows.
// `splits` > 1 cuts K over gridDim.z (not with the gated epilogue; any count that leaves every part 128 of K on average and no part without): `partial` then holds splits * M * N floats, summed
// in ascending order of the split by the other tiled kernel's reduction, which also makes the RMSNorm of the new rows where
// `norm_rows` is given (as there). Returns 0 when it ran, 1 when the shape is not one it takes, -1 on errors.
extern "C" int jllm_gemm_pingpong_bf16(const void* A, int lda, const void* W, const void* W2, const void* bias,
                                       int bias_dtype, void* out, int out_dtype, int ldo, int M, int N, int K,
                                       int epilogue, float gate_limit, int tile_rows, int splits, float* partial, const void* norm_gain,
                                       int norm_gain_dtype, float norm_eps, void* norm_rows, int norm_ld, hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (K < 128 || (K % 32) || (lda & 7)) return 1;
  if (((uintptr_t)A & 15) || ((uintptr_t)W & 15) || (W2 && ((uintptr_t)W2 & 15))) return 1;
  JLLM_TAKE_GATE("gemm_pingpong", epilogue, gate_limit, gs);
  if (epilogue < 0 || epilogue > 2 || (epilogue == 2) != (W2 != nullptr)) JLLM_FAIL("gemm_pingpong: epilogue %d", epilogue);
  if (epilogue == 1 && out_dtype != JLLM_F32) JLLM_FAIL("gemm_pingpong: the accumulate epilogue adds into fp32");
  if (ldo < N) JLLM_FAIL("gemm_pingpong: ldo %d < N %d", ldo, N);
  // a lane's place in an operand is a 32-bit byte offset from the operand's start
  if ((unsigned long long)M * (unsigned)lda * 2ull >= (1ull << 32) || (unsigned long long)N * (unsigned)K * 2ull >= (1ull << 32)) return 1;
  if (splits < 1) splits = 1;
  if (splits > 1 && (W2 || !partial)) JLLM_FAIL("gemm_pingpong: %d K splits are not possible here", splits);
  if (norm_rows && splits == 1) JLLM_FAIL("gemm_pingpong: the norm is the reduction's, and K is whole");
  // (an uneven cut: the last part is what the others, rounded up to whole stages, leave)
  const int stages = (K + PP_BK - 1) / PP_BK, per = (stages + splits - 1) / splits;
  if (splits > 65535 || K / splits < 128 || stages <= per * (splits - 1)) return 1;
  int rc;
  if (tile_rows == 256)
    rc = launch_pingpong<4>(A, lda, W, W2, bias, bias_dtype, out, out_dtype, ldo, M, N, K, epilogue, gs, splits, partial, stream);
  else if (tile_rows == 192)
    rc = launch_pingpong<3>(A, lda, W, W2, bias, bias_dtype, out, out_dtype, ldo, M, N, K, epilogue, gs, splits, partial, stream);
  else if (tile_rows == (256 | 128) && M % 256 >= 1 && M % 256 <= 128)
    rc = launch_mixed(A, lda, W, W2, bias, bias_dtype, out, out_dtype, ldo, M, N, K, epilogue, gs, splits, partial, stream);
  else
    JLLM_FAIL("gemm_pingpong: tile of %d rows for %d (256 and 192 are built; 384: 256 and, where the last rows are at most 128, wide ones for them)", tile_rows, M);
  if (rc != 0) return rc;
  JLLM_CHECK_LAUNCH("gemm_pingpong");
  if (splits > 1 && norm_rows)
    return jllm_splitk_reduce_norm(partial, splits, bias, bias_dtype, out, out_dtype, ldo, M, N, epilogue, norm_gain, norm_gain_dtype, norm_eps, norm_rows, norm_ld, stream);
  if (splits > 1) return jllm_splitk_reduce(partial, splits, bias, bias_dtype, out, out_dtype, ldo, M, N, epilogue, stream);
  return 0;
}
