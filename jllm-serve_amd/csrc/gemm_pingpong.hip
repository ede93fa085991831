// out[M,N] = A[M,K] * W[N,K]^T for many rows, bf16 on the matrix cores (v_mfma_f32_16x16x32_bf16), built so that the
// matrix cores of a compute unit never wait for operands:
//
//  * A workgroup of 8 waves (2 x 4; 1 x 8 for the wide tiles further down) owns a 256 x 256 output tile (a wave 128 x 64: 8 by 4 accumulators of 16 x 16). K
//    advances in stages of 32 through a ring of NS stages in LDS. (The 16 x 16 x 32 form rather than 32 x 32 x 16: the
//    full chip is bound by its power, and a multiply-add of the smaller form reads and writes half as many accumulator
//    bytes. MFMAs alone on random operands run at 2.04 PFLOP/s against 1.85; this kernel with either form: 2,048 rows of
//    the 8B shape's gate/up 340 -> 329 us, qkv 109 -> 103, down 201 -> 188, 8,192^3 923 -> 866 (1.27 PFLOP/s).)
//  * Global -> LDS without registers: global_load_lds_dwordx4 writes 16 bytes per lane straight into LDS, 1 KB
//    (16 tile rows of 64 bytes) per instruction, NS - 1 stages ahead of the multiplies. A lane's place in LDS is
//    fixed by its number, so the bank swizzle is applied on the global side: the lane that fills slot s of row r
//    fetches the row's 16-byte piece s ^ f(r).
//  * The waves form two groups, one wave of each on every SIMD, that run half a stage apart: while one group
//    multiplies (32 MFMAs from registers, nothing else), the other reads the next stage's fragments from LDS and
//    issues its share of the global loads; a workgroup barrier after every phase keeps them apart. A SIMD's matrix
//    core so always has a wave with all operands in registers.
//
// Phases are the times between two workgroup barriers. In phase 2t group 0 is in its memory phase of stage t (it reads
// the second half of the stage's row fragments from LDS and issues the loads of stage t + NS - 1) while group 1 multiplies
// stage t - 1 and, between the multiplies, reads the rest of stage t's fragments; in phase 2t + 1 the groups
// have swapped (group 0 multiplies stage t and reads the first fragments of stage t + 1). So stage s is read from phase
// 2s - 1 on and must have landed when that phase starts: before the barrier in front of it every wave waits until
// its own loads of stages <= s are complete (loads complete in order; group 0 has issued two stages beyond s by
// then, group 1 one). The loads of stage t + NS - 1 go to the slot of stage t - 1, whose last reader (group 1, second
// half, phase 2t - 1) has waited for its LDS reads before the barrier that ends that phase.
//
// A second tile has 192 rows (a wave 96 x 64): it moves a sixth more bytes per multiply and reaches about 0.86 of the rate
// of the 256-row tile (a full chip's stage 0.69 us for 0.75 of the multiplies of one of 0.81 us), but 900 rows of the 8B
// shape's gate/up are 480 tiles in two rounds of 256 compute units instead of 384 in two: 196 -> 177 us.
//
// Epilogues as in the other tiled kernel (gemm_epilogue.h). Needs K % 32 == 0 and at least NS - 1 stages, 16-byte
// aligned rows; any M and N (rows beyond the end are read as the last row and never stored).
#include "common.h"
#include "layer_launches.h"
#include "lds_ring.h"
#include "gemm_epilogue.h"
#include "mfma.h"

#define PP_BK 32
#define PP_ROW_BYTES (PP_BK * 2)  // a tile row in LDS: 64 bytes = 4 pieces of 16
#define PP_WAVES 8

// The piece of row r that lies in slot s is s ^ pp_swz(r): 16 lanes that read the same piece of 16 consecutive rows,
// and 8 lanes of 8 rows, then cover every bank once, whichever of the two the LDS takes per pass. (With fragments of 32 rows
// the counter shows no conflict; with these of 16 rows and four pieces four cycles per LDS instruction.)
__device__ __forceinline__ int pp_swz(int r) { return (((r >> 1) ^ (r >> 3)) & 1) | (((r >> 2) & 1) << 1); }

#define PP_VMCNT(n) __builtin_amdgcn_s_waitcnt(((n) & 15) | (((n) >> 4) << 14) | (7 << 4) | (15 << 8))
#define PP_LGKMCNT0() __builtin_amdgcn_s_waitcnt((15) | (3 << 14) | (7 << 4) | (0 << 8))

// WGM x 8 / WGM waves of 32 FM rows by 64 columns each: the tile whose first row and first output are m0 and n0
template <bool GATED, int FM, int NS, int WGM>
__device__ __forceinline__ void pingpong_tile(
    const bf16_t* __restrict__ A, int lda, const bf16_t* __restrict__ W, const bf16_t* __restrict__ W2,
    const void* __restrict__ bias, int bias_dtype, void* __restrict__ out, int out_dtype, int ldo, int M, int N, int K,
    int epilogue, GateSpec gs, float* __restrict__ partial, int m0, int n0) {
  constexpr int WGN = PP_WAVES / WGM, RM = 2 * FM, CN = 4;  // a wave's blocks of 16 rows and of 16 columns
  constexpr int TBM = WGM * RM * 16, TBN = WGN * CN * 16;
  constexpr int STAGE = (TBM + TBN) * PP_ROW_BYTES;
  // load instructions (16 rows each) per wave and stage. Tiles of 192 rows are twelve chunks of A: two for each wave of the
  // first group, one for each of the second's.
  constexpr int LA = (TBM / 16 + PP_WAVES - 1) / PP_WAVES, LB = TBN / 16 / PP_WAVES, LA1 = TBM / 16 * 2 / PP_WAVES - LA;
  constexpr int L0 = LA + LB, L1 = LA1 + LB;
  static_assert(LA1 >= 0 && LB >= 1 && (LA + LA1) * PP_WAVES / 2 == TBM / 16, "every wave loads rows of both operands");
  extern __shared__ __align__(1024) unsigned char smem[];
  const int tid = threadIdx.x;
  // the wave's number is the same in all its lanes: said so, its group, its part of the tile and the places in LDS it
  // fills stay in scalar registers (no vector arithmetic for them per stage, jumps instead of lane masks)
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int group = wave >> 2;  // waves 0..3 and 4..7: one of each on every SIMD
  const int wm = wave / WGN, wn = wave % WGN;
  const int nk_all = K / PP_BK;
  const int nk_per = (nk_all + gridDim.z - 1) / gridDim.z;
  const int kt0 = blockIdx.z * nk_per;
  const int nk = max(0, min(nk_all, kt0 + nk_per) - kt0);

  // ---- global side of the loads: this lane's piece of each of the wave's 16-row chunks. The address of a load is a
  // scalar base (the operand's start plus the stage's place in K, advanced by scalar arithmetic) plus a 32-bit byte
  // offset per lane that never changes (row and piece), so a stage's loads cost no vector instruction.
  const int lrow = lane >> 2, lslot = lane & 3;
  uint32_t goff[L0];               // this lane's byte offset from the operand's start (rows x row length < 4 GB: checked on the host)
  const unsigned char* gbase[L0];  // the operand's start at this workgroup's first K step (the same in all lanes)
  uint32_t ldst[L0];               // LDS byte address of the chunk inside stage 0 (the same in all lanes)
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)smem;
#pragma unroll
  for (int c = 0; c < LA; ++c) {
    const int chunk = LA == LA1 || group == 0 ? wave * LA + c : PP_WAVES / 2 * LA + (wave - PP_WAVES / 2) * LA1;  // (the second group's c = LA1 .. is never asked for)
    const int r = chunk * 16 + lrow;
    goff[c] = (uint32_t)min(m0 + r, M - 1) * (uint32_t)lda * 2u + (uint32_t)((lslot ^ pp_swz(r)) * 16);
    gbase[c] = (const unsigned char*)A + (size_t)kt0 * PP_ROW_BYTES;
    ldst[c] = lds0 + chunk * 16 * PP_ROW_BYTES;
  }
#pragma unroll
  for (int c = 0; c < LB; ++c) {
    const int r = (wave * LB + c) * 16 + lrow;
    int wr;
    const bf16_t* wb = W;
    if (GATED) {  // LDS row r: quarter r / 32: even = gate, odd = up of the outputs n0 + (quarter / 2) * 32 ..
      const int quarter = (wave * LB + c) >> 1;  // of the chunk's 16 rows: the same in all lanes
      wr = n0 + (quarter >> 1) * 32 + (r & 31);
      wb = (quarter & 1) ? W2 : W;
    } else {
      wr = n0 + r;
    }
    goff[LA + c] = (uint32_t)min(wr, N - 1) * (uint32_t)K * 2u + (uint32_t)((lslot ^ pp_swz(r)) * 16);
    gbase[LA + c] = (const unsigned char*)wb + (size_t)kt0 * PP_ROW_BYTES;
    ldst[LA + c] = lds0 + TBM * PP_ROW_BYTES + (wave * LB + c) * 16 * PP_ROW_BYTES;
  }
  auto issue = [&](int t) {  // the wave's loads of stage t
    const uint32_t slot = (uint32_t)(t % NS) * STAGE;
    const size_t kbytes = (size_t)t * PP_ROW_BYTES;
#pragma unroll
    for (int c = 0; c < L0; ++c) {
      if (c >= LA1 && c < LA && group != 0) continue;
      load_to_lds_16(gbase[c] + kbytes, goff[c], ldst[c] + slot);
    }
  };

  // ---- LDS side: fragment of a block of 16 rows: row = block * 16 + lane % 16, piece = lane / 16 (16 bytes: 8 of the stage's k)
  const int ra = wm * RM * 16 + (lane & 15), rb = wn * CN * 16 + (lane & 15);  // + 16 i leaves pp_swz unchanged
  const int aoff = ra * PP_ROW_BYTES + (((lane >> 4) ^ pp_swz(ra)) * 16);
  const int boff = TBM * PP_ROW_BYTES + rb * PP_ROW_BYTES + (((lane >> 4) ^ pp_swz(rb)) * 16);

  floatx4 acc[RM][CN];
#pragma unroll
  for (int i = 0; i < RM; ++i)
#pragma unroll
    for (int j = 0; j < CN; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};

  // ---- prologue: NS - 1 stages on their way, stages 0 and 1 landed
#pragma unroll
  for (int s = 0; s < NS - 1; ++s)
    if (s < nk) issue(s);
  if (nk < NS - 1) {
    PP_VMCNT(0);
  } else if (group == 0) {
    PP_VMCNT((NS - 3) * L0);
  } else {
    PP_VMCNT((NS - 3) * L1);
  }
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
  // fragments of a stage: the weights' and the first half of the rows' (read during the multiplies of the stage before), the
  // second half of the rows' (read in the memory phase); the loop is unrolled by two so that a stage's and the next
  // one's swap names instead of being copied
  constexpr int RH = RM / 2;
  constexpr int PP_MUL = RM > 4 ? 3 : 2;  // multiplies between two LDS reads of the multiply phase
  u32x4 a0[RH], b0[CN], a1[RH], an[RH], bn[CN];
  auto read_rows = [&](int t, int half, u32x4 (&af)[RH]) {
    const unsigned char* st = smem + (t % NS) * STAGE + aoff + half * RH * 16 * PP_ROW_BYTES;
#pragma unroll
    for (int i = 0; i < RH; ++i) af[i] = *(const u32x4*)(st + i * 16 * PP_ROW_BYTES);
  };
  auto read_cols = [&](int t, u32x4 (&bf)[CN]) {
    const unsigned char* st = smem + (t % NS) * STAGE + boff;
#pragma unroll
    for (int j = 0; j < CN; ++j) bf[j] = *(const u32x4*)(st + j * 16 * PP_ROW_BYTES);
  };
  // one stage of one group. Memory phase: the second half of the rows' fragments, then the global loads (a compute
  // unit's load pipe takes about 40 cycles per load instruction and a wave waits at the issue while it is busy, so
  // the LDS reads go first). Multiply phase: 32 MFMAs with the reads of the next stage's first fragments between them.
  auto stage = [&](int t, u32x4 (&fa0)[RH], u32x4 (&fb0)[CN], u32x4 (&na0)[RH], u32x4 (&nb0)[CN]) {
    const bool more = t + NS - 1 < nk;
    read_rows(t, 1, a1);
    __builtin_amdgcn_sched_barrier(0);
    if (more) issue(t + NS - 1);
    // own loads of stage t + 1 must have landed before the barrier that lets group 0 read it during its multiplies:
    // group 0 is here (it has issued up to stage t + 3), group 1 at the end of its multiplies of stage t - 1
    if (group == 0) {
      if (more) {
        PP_VMCNT(2 * L0);
      } else {
        PP_VMCNT(0);
      }
    }
    PP_LGKMCNT0();
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    read_cols(t + 1, nb0);  // beyond the last stage: some slot's bytes, never multiplied
    read_rows(t + 1, 0, na0);
#pragma unroll
    for (int i = 0; i < RH; ++i)
#pragma unroll
      for (int j = 0; j < CN; ++j) acc[i][j] = mfma16(fb0[j], fa0[i], acc[i][j]);
#pragma unroll
    for (int i = 0; i < RH; ++i)
#pragma unroll
      for (int j = 0; j < CN; ++j) acc[RH + i][j] = mfma16(fb0[j], a1[i], acc[RH + i][j]);
    // order of issue: PP_MUL multiplies, then one LDS read, ...; the rest of the multiplies
#pragma unroll
    for (int r = 0; r < RH + CN; ++r) {
      __builtin_amdgcn_sched_group_barrier(0x008, PP_MUL, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x008, RM * CN - PP_MUL * (RH + CN), 0);
    if (group == 1) {  // has issued up to stage t + 3; stage t + 2 must have landed (group 0 reads it after the next barrier but one)
      if (more) {
        PP_VMCNT(1 * L1);
      } else {
        PP_VMCNT(0);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
  };
  if (nk > 0) {
    read_cols(0, b0);
    read_rows(0, 0, a0);
  }
  if (group == 1) {  // half a stage behind
    PP_LGKMCNT0();
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
  }
  for (int t = 0; t < nk; t += 2) {
    stage(t, a0, b0, an, bn);
    if (t + 1 < nk) stage(t + 1, an, bn, a0, b0);
  }
  if (group == 0) {  // as many barriers as the other group
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
  }
  tile_epilogue<GATED, 16, RM, CN, TBM, TBN>(acc, lane, wm, wn, m0, n0, bias, bias_dtype, out, out_dtype, ldo, M, N, epilogue, gs, partial,
                                         (int)blockIdx.z, (int)gridDim.z);
}

template <bool GATED, int FM, int NS>
__global__ __launch_bounds__(PP_WAVES * 64) void gemm_pingpong_kernel(
    const bf16_t* __restrict__ A, int lda, const bf16_t* __restrict__ W, const bf16_t* __restrict__ W2,
    const void* __restrict__ bias, int bias_dtype, void* __restrict__ out, int out_dtype, int ldo, int M, int N, int K,
    int epilogue, GateSpec gs, float* __restrict__ partial) {
  pingpong_tile<GATED, FM, NS, 2>(A, lda, W, W2, bias, bias_dtype, out, out_dtype, ldo, M, N, K, epilogue, gs, partial,
                                  blockIdx.y * 64 * FM, blockIdx.x * (GATED ? 128 : 256));
}

// Tiles of 256 x 256 and, for the last rows where those are at most 128, of 128 x 512 (64 x 512 where they are at most 64): `wide`
// of the latter, which come first because they take longer, then rows of `cols` of the former. A tile of 256 rows of which a few
// are there takes as long as a full one, and so does the round of workgroups that it begins. A wide tile takes half as many
// workgroups; its stage moves a quarter (an eighth) more bytes into LDS and takes 1.25 (1.17) times as long. us, what was chosen
// among whole tiles / this: gate/up of the 8B shape at 560 rows (288 tiles / 240) 167 / 122, at 631 171 / 131, of the 14B shape at 300 223 / 153,
// at 1,320 522 / 457, at 4,614 (10.1 rounds / 9.8) 1,558 / 1,498, of the 32B shape at 600 412 / 345; 14B down at 3,111 620 / 501, 4B
// qkv at 2,600 106 / 75. Last rows of 129 to 192 in a tile of either kind gained nothing (8B gate/up at 700 rows 169 / 196).
template <bool GATED, int NS>
__global__ __launch_bounds__(PP_WAVES * 64) void gemm_pingpong_mixed_kernel(
    const bf16_t* __restrict__ A, int lda, const bf16_t* __restrict__ W, const bf16_t* __restrict__ W2,
    const void* __restrict__ bias, int bias_dtype, void* __restrict__ out, int out_dtype, int ldo, int M, int N, int K,
    int epilogue, GateSpec gs, float* __restrict__ partial, int wide, int cols) {
  const int whole = M >> 8 << 8, b = blockIdx.x;
  if (b >= wide) {
    const int row = (b - wide) / cols, col = b - wide - row * cols;
    pingpong_tile<GATED, 4, NS, 2>(A, lda, W, W2, bias, bias_dtype, out, out_dtype, ldo, M, N, K, epilogue, gs, partial, row * 256, col * (GATED ? 128 : 256));
  } else if (M - whole > 64) {
    pingpong_tile<GATED, 4, NS, 1>(A, lda, W, W2, bias, bias_dtype, out, out_dtype, ldo, M, N, K, epilogue, gs, partial, whole, b * (GATED ? 256 : 512));
  } else {
    pingpong_tile<GATED, 2, NS, 1>(A, lda, W, W2, bias, bias_dtype, out, out_dtype, ldo, M, N, K, epilogue, gs, partial, whole, b * (GATED ? 256 : 512));
  }
}

template <int FM, int NS>
static int launch_pingpong(const void* A, int lda, const void* W, const void* W2, const void* bias, int bias_dtype,
                           void* out, int out_dtype, int ldo, int M, int N, int K, int epilogue, GateSpec gs, int splits,
                           float* partial, hipStream_t stream) {
  constexpr int TBM = 4 * FM * 16, TBN = 256;
  const int cols = W2 ? TBN / 2 : TBN;
  dim3 grid((N + cols - 1) / cols, (M + TBM - 1) / TBM, splits);
  if (grid.y > 65535) return 1;
  const size_t smem = (size_t)NS * (TBM + TBN) * PP_ROW_BYTES;
  static bool configured = false;
  if (!configured) {
    hipError_t e1 = hipFuncSetAttribute((const void*)gemm_pingpong_kernel<true, FM, NS>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
    hipError_t e2 = hipFuncSetAttribute((const void*)gemm_pingpong_kernel<false, FM, NS>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
    if (e1 != hipSuccess || e2 != hipSuccess) JLLM_FAIL("gemm_pingpong: cannot reserve %zu bytes of LDS", smem);
    configured = true;
  }
  if (W2)
    gemm_pingpong_kernel<true, FM, NS><<<grid, PP_WAVES * 64, smem, stream>>>(
        (const bf16_t*)A, lda, (const bf16_t*)W, (const bf16_t*)W2, bias, bias_dtype, out, out_dtype, ldo, M, N, K, epilogue, gs, partial);
  else
    gemm_pingpong_kernel<false, FM, NS><<<grid, PP_WAVES * 64, smem, stream>>>(
        (const bf16_t*)A, lda, (const bf16_t*)W, nullptr, bias, bias_dtype, out, out_dtype, ldo, M, N, K, epilogue, gs, partial);
  return 0;
}

static int launch_mixed(const void* A, int lda, const void* W, const void* W2, const void* bias, int bias_dtype,
                        void* out, int out_dtype, int ldo, int M, int N, int K, int epilogue, GateSpec gs, int splits,
                        float* partial, hipStream_t stream) {
  constexpr int NS = 4;
  const int cols = (N + (W2 ? 127 : 255)) / (W2 ? 128 : 256), wide = (cols + 1) / 2;
  const long groups = (long)(M / 256) * cols + wide;
  if (groups > 0x7fffffffl) return 1;
  constexpr size_t smem = (size_t)NS * (128 + 512) * PP_ROW_BYTES;  // of the wider stage
  static bool configured = false;
  if (!configured) {
    hipError_t e1 = hipFuncSetAttribute((const void*)gemm_pingpong_mixed_kernel<true, NS>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
    hipError_t e2 = hipFuncSetAttribute((const void*)gemm_pingpong_mixed_kernel<false, NS>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
    if (e1 != hipSuccess || e2 != hipSuccess) JLLM_FAIL("gemm_pingpong: cannot reserve %zu bytes of LDS", smem);
    configured = true;
  }
  dim3 grid((unsigned)groups, 1, splits);
  if (W2)
    gemm_pingpong_mixed_kernel<true, NS><<<grid, PP_WAVES * 64, smem, stream>>>(
        (const bf16_t*)A, lda, (const bf16_t*)W, (const bf16_t*)W2, bias, bias_dtype, out, out_dtype, ldo, M, N, K, epilogue, gs, partial, wide, cols);
  else
    gemm_pingpong_mixed_kernel<false, NS><<<grid, PP_WAVES * 64, smem, stream>>>(
        (const bf16_t*)A, lda, (const bf16_t*)W, nullptr, bias, bias_dtype, out, out_dtype, ldo, M, N, K, epilogue, gs, partial, wide, cols);
  return 0;
}

// `tile_rows`: 256 or 192 (rows of the output tile; 256 columns, 128 outputs with the gated epilogue), or 384: tiles of 256 rows and
// wide ones for the last at most 128 rows.
// `splits` > 1 cuts K over gridDim.z (not with the gated epilogue; any count that leaves every part four stages): `partial` then holds splits * M * N floats, summed
// in ascending order of the split by the other tiled kernel's reduction, which also makes the RMSNorm of the new rows where
// `norm_rows` is given (as there). Returns 0 when it ran, 1 when the shape is not one it takes, -1 on errors.
extern "C" int jllm_gemm_pingpong_bf16(const void* A, int lda, const void* W, const void* W2, const void* bias,
                                       int bias_dtype, void* out, int out_dtype, int ldo, int M, int N, int K,
                                       int epilogue, float gate_limit, int tile_rows, int splits, float* partial, const void* norm_gain,
                                       int norm_gain_dtype, float norm_eps, void* norm_rows, int norm_ld, hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (K <= 0 || (K % PP_BK) || (lda & 7)) return 1;
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
  if (splits > 65535 || (K / PP_BK) / splits < 4) return 1;
  // (an uneven cut: the last part is what the others, rounded up, leave)
  const int per = (K / PP_BK + splits - 1) / splits;
  if (K / PP_BK - per * (splits - 1) < 4) return 1;
  int rc;
  if (tile_rows == 256)
    rc = launch_pingpong<4, 4>(A, lda, W, W2, bias, bias_dtype, out, out_dtype, ldo, M, N, K, epilogue, gs, splits, partial, stream);
  else if (tile_rows == 192)
    rc = launch_pingpong<3, 4>(A, lda, W, W2, bias, bias_dtype, out, out_dtype, ldo, M, N, K, epilogue, gs, splits, partial, stream);
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
