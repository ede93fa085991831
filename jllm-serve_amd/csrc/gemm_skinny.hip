// out[M,N] = A[M,K] * W[N,K]^T for up to 16 rows (decode steps): bf16 operands, fp32 accumulation on the matrix cores
// (16x16x32), bound by streaming W from HBM once.
//
// A workgroup of 8 (or 4) waves owns `rows` weight rows (up to 32, 16 with the gated epilogue) and cuts K, in blocks of
// 64, among its waves: wave w takes blocks w, w + WAVES, ... Both operands of a block go straight from memory into a ring
// of S blocks in LDS that belongs to the wave alone (global_load_lds_dwordx4, 1 KB per instruction: 8 rows of 128 bytes),
// S - 1 blocks ahead of the multiplies; nothing but the wave's own counter of loads in flight stands between a load and its
// use, so there is no barrier before the end. A lane's place in LDS is fixed by its number, so the bank swizzle is
// applied on the global side: the lane that fills slot s of row r fetches the row's 16-byte piece s ^ ring_swz(r).
//
// Why not from memory into the registers that feed the matrix cores, as this kernel used to: such a load takes 64 bytes of
// each of 16 rows, and a compute unit's load pipe then passes 25 bytes a clock (6.6 TB/s of the whole chip with everything in
// L2, against 10 for 8 rows of 128 bytes), which the activations, once per workgroup and as many as the weights at 16 rows,
// had to share. In LDS the activations of up to 8 rows cost half as much, and K blocks of 64 keep the waves even.
// Inside a graph, before / now, in us at 1, 8 and 16 rows: 8B shape qkv 13.9 15.6 16.1 / 11.6 12.9 13.1, o 8.7 9.8 11.3 / 8.3
// 8.7 9.4, gate/up 40.1 41.4 45.6 / 37.2 38.4 39.1, down 20.9 25.2 30.6 / 20.2 21.0 23.1; 32B down 52.3 61.5 71.5 / 48.8 50.1
// 52.9; 0.6B o 4.7 5.7 6.4 / 4.0 4.4 4.7, down 7.4 9.1 10.4 / 4.8 5.4 5.9; 1.7B qkv 6.0 7.2 7.6 / 6.0 6.8 7.1.
// What a large copy reaches (6.2 TB/s) would take 8.1, 5.4, 32.5 and 16.2 us of the 8B shape's four: what is left is the
// launch, the first bytes' latency and the sum over the waves, about 4 us each. Measured and not taken: three blocks in
// flight instead of up to six (8B gate/up at one row 37.9 -> 38.2), a contiguous range of K per wave (42.2).
//
// The WAVES partial tiles are summed through LDS in wave order, and how K is cut depends on nothing but K and N: a row's
// result depends neither on M nor on the rows beside it.
//
// How many weight rows a workgroup owns (`rows`) is the caller's choice: as many as let N / rows workgroups fill the
// compute units evenly. Rows beyond those (a load covers eight) are the last row again and never stored.
//
// An RMSNorm between two such products costs no launch of its own. The product that adds into the residual
// ("emit") also leaves, for the norm that follows, the new residual values times that norm's gain as bf16
// [M, N] and the sum of their squares over its columns as partial[m][block]. The product that consumes the
// norm ("normed") takes those bf16 rows as its input and multiplies its sums by rsqrt(sum of the partials / K +
// eps) at the end: sum_k W[n,k] (x[k] g[k]) s = the product over the normalised row. The partials are summed in
// an order that depends on nothing but their count.
//
// Needs K % 128 == 0, N % 16 == 0, M <= 16, 16-byte aligned rows; the caller falls back otherwise.
#include "common.h"
#include "layer_launches.h"
#include "lds_ring.h"
#include "mfma.h"

#define SK_BLOCK 64                    // k per block
#define SK_ROW_BYTES (SK_BLOCK * 2)    // a row of a block in LDS: 128 bytes = 8 pieces of 16

// what the two norm-carrying forms need beyond the plain product
struct SkinnyNorm {
  bf16_t* emit_rows;          // emit: [M, N] bf16, (residual after the add) * emit_gain
  const void* emit_gain;      // [N]
  int emit_gain_dtype;
  float* emit_partial;        // [M][emit_parts]: a sum per workgroup, zeros behind them
  int emit_parts;
  const float* norm_partial;  // normed: [M][norm_parts] sums of squares of the input rows
  int norm_parts;
  float norm_eps;
  GateSpec gate;              // the gate function of the gated epilogue
};

// sum over the 16 lanes of a row of lanes (the 16 columns of a tile), left in all of them
__device__ __forceinline__ float row16_sum(float d) {
  d += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, d), 0xB1, 0xF, 0xF, true));
  d += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, d), 0x4E, 0xF, 0xF, true));
  d += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, d), 0x141, 0xF, 0xF, true));
  d += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, d), 0x140, 0xF, 0xF, true));
  return d;
}

// NI loads per block: a ring as deep as the LDS allows, with `per_cu` workgroups on a compute unit
constexpr int sk_slots(int ni, int waves, int per_cu) {
  const int fit = (160 / per_cu - 1) / (waves * ni);
  return fit > 6 ? 6 : fit;
}

template <int NI, int S>
__device__ __forceinline__ void sk_wait_block(int behind) {  // `behind` (< S) blocks behind the one that has to be here
  if (behind == S - 1) return wait_loads<(S - 1) * NI>();
  if (S > 2 && behind == S - 2) return wait_loads<(S > 2 ? S - 2 : 0) * NI>();
  if (S > 3 && behind == S - 3) return wait_loads<(S > 3 ? S - 3 : 0) * NI>();
  if (S > 4 && behind == S - 4) return wait_loads<(S > 4 ? S - 4 : 0) * NI>();
  if (S > 5 && behind == S - 5) return wait_loads<(S > 5 ? S - 5 : 0) * NI>();
  wait_loads<0>();
}

// NW: loads of 8 weight rows per block (of each weight), NA: of 8 activation rows; TURN: see the host's rule
template <int NW, int NA, bool GATED, int WAVES, int PER_CU, bool TURN>
__global__ __launch_bounds__(WAVES * 64) void gemm_skinny_kernel(
    const bf16_t* __restrict__ A, const bf16_t* __restrict__ W, const bf16_t* __restrict__ W2, int lda, int M, int N, int K, int rows,
    int epilogue, const void* __restrict__ bias, int bias_dtype, void* __restrict__ out, int out_dtype, int ldo, SkinnyNorm nm) {
  constexpr int CT = (NW + 1) / 2;                // tiles of 16 weight rows
  constexpr int TILES = GATED ? 2 : CT;           // accumulators: gate and up, or the weight's tiles
  constexpr int NI = (GATED ? 2 : 1) * NW + NA;   // loads of a block
  constexpr int S = sk_slots(NI, WAVES, PER_CU);
  static_assert(!GATED || CT == 1, "the gated epilogue takes up to 16 rows of each weight");
  static_assert(S >= 2 && (S - 1) * NI < 63, "the counter of loads in flight");
  extern __shared__ __align__(1024) unsigned char smem[];   // [WAVES][S][NI KB]; afterwards the waves' sums
  __shared__ float ssq[WAVES][16];                          // normed: each wave's share of the rows' sums of squares
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int col = lane & 15;
  const int g = lane >> 4;
  const int n0 = blockIdx.x * rows;
  const int nblk = K / SK_BLOCK;
  // gated: workgroups walk K from different starting blocks, so that at any moment they ask the L2 for different parts of
  // the (shared) activations (12,288 x 4,096 at one row 39.2 -> 37.9 us); without the gate from a power of two of them
  // (which needs no division) where the host says so
  const int rot = GATED  ? (int)((blockIdx.x * 14u) % (unsigned)nblk)
                  : TURN ? (int)(blockIdx.x & ((1u << (31 - __builtin_clz((unsigned)nblk))) - 1u))
                         : 0;
  // Wave 0 writes the outputs: what it adds into (the residual, the bias) is requested before anything else, as it lies in memory
  // and from rows that are there: a conversion, or a branch of single lanes, waits for its load before the next request goes out,
  // and wave 0 begins its share of K two latencies behind the others: 0.8 us a launch of the two in each layer that add (a step of
  // 300 keys of the 0.6B shape 875 -> 831 us, four of 6,100 to 8,000 keys (4B) 3,028 -> 2,970; 8B, whose rows are longer, as before).
  float prev[CT][4];
  uint32_t raw_b[CT], raw_eg[CT];
#pragma unroll
  for (int t = 0; t < CT; ++t) {
    raw_b[t] = raw_eg[t] = 0u;
#pragma unroll
    for (int i = 0; i < 4; ++i) prev[t][i] = 0.f;
  }
  if (wave == 0) {
#pragma unroll
    for (int t = 0; t < CT; ++t) {
      const int n = min(n0 + min(t * 16 + col, rows - 1), N - 1);
      if (bias) raw_b[t] = raw_entry(bias, bias_dtype, n);
      if (nm.emit_rows) raw_eg[t] = raw_entry(nm.emit_gain, nm.emit_gain_dtype, n);
      if (epilogue == 1) {
#pragma unroll
        for (int i = 0; i < 4; ++i) prev[t][i] = ((const float*)out)[(size_t)min(g * 4 + i, M - 1) * ldo + n];
      }
    }
  }
  // normed: the sums of squares of the input rows. Every wave takes a share: lane `col` of wave w the four partials
  // 4 (16 w + col) .., requested here and added up behind the products, then those 64 WAVES further on
  floatx4 first[4];
  if (nm.norm_partial) {
    const int p4 = min(wave * 16 + col, (nm.norm_parts >> 2) - 1);
    first[0] = ((const floatx4*)(nm.norm_partial + (size_t)min(g * 4, M - 1) * nm.norm_parts))[p4];
    if (M > 1) {
#pragma unroll
      for (int i = 1; i < 4; ++i) first[i] = ((const floatx4*)(nm.norm_partial + (size_t)min(g * 4 + i, M - 1) * nm.norm_parts))[p4];
    }
  }
  // ---- the loads of a block: a scalar base that advances with the block and a byte offset per lane that never changes
  uint32_t goff[NI];
  const int lrow = lane >> 3, lslot = lane & 7;
#pragma unroll
  for (int c = 0; c < NI; ++c) {
    const bool of_w = c < NI - NA;
    const int r = (of_w ? c % NW : c - (NI - NA)) * 8 + lrow;
    const uint32_t at = of_w ? (uint32_t)(min(n0 + min(r, rows - 1), N - 1) - n0) * (uint32_t)K : (uint32_t)min(r, M - 1) * (uint32_t)lda;
    goff[c] = at * 2u + (uint32_t)((lslot ^ ring_swz(r)) * 16);
  }
  const unsigned char* wbase = (const unsigned char*)(W + (size_t)n0 * K);
  const unsigned char* ubase = GATED ? (const unsigned char*)(W2 + (size_t)n0 * K) : nullptr;
  const unsigned char* ring = smem + (size_t)wave * S * NI * 1024;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const unsigned char*)ring;
  const int total = wave < nblk ? (nblk - wave + WAVES - 1) / WAVES : 0;
  auto issue = [&](int i, int slot) {
    int bb = wave + i * WAVES + rot;
    if (bb >= nblk) bb -= nblk;
    const size_t kbytes = (size_t)bb * SK_ROW_BYTES;
#pragma unroll
    for (int c = 0; c < NI; ++c) {
      const unsigned char* base = (c >= NI - NA ? (const unsigned char*)A : GATED && c >= NW ? ubase : wbase) + kbytes;
      load_to_lds_16(base, goff[c], lds0 + (uint32_t)(slot * NI + c) * 1024u);
    }
  };
#pragma unroll
  for (int i = 0; i < S; ++i)
    if (i < total) issue(i, i);
  // ---- fragments: lane l reads row l % 16, 8 of k at (l / 16) * 8 + 32 j: piece l / 16 + 4 j. Rows that no load fetched
  // (eight activation rows, up to eight weight rows in a tile) are the last fetched eight again.
  const int ar = NA == 1 ? col & 7 : col;
  const int aoff = ((GATED ? 2 : 1) * NW) * 1024 + ar * SK_ROW_BYTES, aswz = ring_swz(ar);
  int woff[TILES], wswz[TILES];
#pragma unroll
  for (int t = 0; t < TILES; ++t) {
    const int left = GATED ? NW : NW - 2 * t;  // loads that this tile has
    const int r = (GATED ? 0 : t * 16) + (left == 1 ? col & 7 : col);
    woff[t] = (GATED ? t * NW * 1024 : 0) + r * SK_ROW_BYTES;
    wswz[t] = ring_swz(r);
  }
  floatx4 acc[TILES];
#pragma unroll
  for (int t = 0; t < TILES; ++t) acc[t] = floatx4{0.f, 0.f, 0.f, 0.f};
  int slot = 0;
  for (int i = 0; i < total; ++i) {
    sk_wait_block<NI, S>(min(S - 1, total - 1 - i));
    const unsigned char* blk = ring + slot * NI * 1024;
    u32x4 a[2], w[TILES][2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      a[j] = *(const u32x4*)(blk + aoff + (((g + 4 * j) ^ aswz) << 4));
#pragma unroll
      for (int t = 0; t < TILES; ++t) w[t][j] = *(const u32x4*)(blk + woff[t] + (((g + 4 * j) ^ wswz[t]) << 4));
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the slot's last reads, before it is filled again
    __builtin_amdgcn_sched_barrier(0);
    if (i + S < total) issue(i + S, slot);
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int t = 0; t < TILES; ++t) acc[t] = mfma16(a[j], w[t][j], acc[t]);
    if (++slot == S) slot = 0;
  }
  // (of one row three in four are no lane's: left out, a normed product of one row takes 0.5 us less; a branch for each of
  // the four made more rows 1 to 2 % slower)
  if (nm.norm_partial) {
    auto squares = [&](int i) {
      float t = wave * 16 + col < nm.norm_parts >> 2 ? (first[i][0] + first[i][1]) + (first[i][2] + first[i][3]) : 0.f;
      if (g * 4 + i < M)
        for (int p4 = (WAVES + wave) * 16 + col; p4 < nm.norm_parts >> 2; p4 += WAVES * 16) {
          const floatx4 v = ((const floatx4*)(nm.norm_partial + (size_t)(g * 4 + i) * nm.norm_parts))[p4];
          t += (v[0] + v[1]) + (v[2] + v[3]);
        }
      t = row16_sum(t);
      if (col == 0) ssq[wave][g * 4 + i] = t;
    };
    squares(0);
    if (M > 1) squares(1), squares(2), squares(3);
  }
  // the sums meet in LDS, in wave order
  __syncthreads();  // every wave is done with its ring
  floatx4(*red)[TILES][64] = (floatx4(*)[TILES][64])smem;
  if (wave > 0) {
#pragma unroll
    for (int t = 0; t < TILES; ++t) red[wave - 1][t][lane] = acc[t];
  }
  __syncthreads();
  if (wave != 0) return;
#pragma unroll
  for (int t = 0; t < TILES; ++t)
#pragma unroll
    for (int w = 0; w < WAVES - 1; ++w) acc[t] += red[w][t][lane];
  float rscale[4];  // normed: rsqrt(mean of squares + eps) of the rows this lane writes
#pragma unroll
  for (int i = 0; i < 4; ++i) rscale[i] = 1.0f;
  if (nm.norm_partial) {
    auto scale = [&](int i) {
      float t = 0.f;
#pragma unroll
      for (int w = 0; w < WAVES; ++w) t += ssq[w][g * 4 + i];
      rscale[i] = 1.0f / sqrtf(t / (float)K + nm.norm_eps);
    };
    scale(0);
    if (M > 1) scale(1), scale(2), scale(3);
  }
  float b[CT], eg[CT];
#pragma unroll
  for (int t = 0; t < CT; ++t) b[t] = raw_value(raw_b[t], bias_dtype), eg[t] = raw_value(raw_eg[t], nm.emit_gain_dtype);
  float sq[4] = {0.f, 0.f, 0.f, 0.f};  // emit: the squares of the workgroup's columns, per row of this lane
#pragma unroll
  for (int t = CT - 1; t >= 0; --t) {
    const int n = n0 + t * 16 + col;
    const bool mine = t * 16 + col < rows && n < N;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int m = g * 4 + i;
      float v = acc[t][i] * rscale[i] + b[t];
      if (GATED) v = gated<false>(v, acc[GATED ? 1 : 0][i] * rscale[i], nm.gate);
      const float now = prev[t][i] + v;
      // every lane of the row takes part in the sum, columns and rows that are not there with zeros
      if (nm.emit_rows) sq[i] = row16_sum(mine && m < M ? now * now : 0.f) + sq[i];
      if (m >= M || !mine) continue;
      const size_t o = (size_t)m * ldo + n;
      if (nm.emit_rows) nm.emit_rows[(size_t)m * N + n] = f32_to_bf16(now * eg[t]);
      if (epilogue == 1)
        ((float*)out)[o] = now;
      else if (out_dtype == JLLM_BF16)
        stf((bf16_t*)out, o, v);
      else
        stf((float*)out, o, v);
    }
  }
  if (nm.emit_rows && col == 0) {
    const int spare = nm.emit_parts - (int)gridDim.x;  // partial sums behind the workgroups' own: zeros
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int m = g * 4 + i;
      if (m >= M) continue;
      nm.emit_partial[(size_t)m * nm.emit_parts + blockIdx.x] = sq[i];
      for (int z = blockIdx.x; z < spare; z += gridDim.x) nm.emit_partial[(size_t)m * nm.emit_parts + gridDim.x + z] = 0.f;
    }
  }
}

struct SkinnyArgs {
  const bf16_t *A, *W, *W2;
  const void* bias;
  int lda, bias_dtype, out_dtype, ldo, M, N, K, epilogue, rows;
  void* out;
};

template <int NW, int NA, bool GATED, int WAVES, int PER_CU, bool TURN>
static int launch_skinny(const SkinnyArgs& a, const SkinnyNorm& nm, hipStream_t stream) {
  constexpr int NI = (GATED ? 2 : 1) * NW + NA;
  constexpr size_t smem = (size_t)sk_slots(NI, WAVES, PER_CU) * WAVES * NI * 1024;
  static bool configured = false;
  if (!configured) {  // above 64 KB the size has to be allowed first
    if (hipFuncSetAttribute((const void*)gemm_skinny_kernel<NW, NA, GATED, WAVES, PER_CU, TURN>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem) != hipSuccess)
      JLLM_FAIL("gemm_skinny: cannot reserve %zu bytes of LDS", smem);
    configured = true;
  }
  gemm_skinny_kernel<NW, NA, GATED, WAVES, PER_CU, TURN><<<(a.N + a.rows - 1) / a.rows, WAVES * 64, smem, stream>>>(
      a.A, a.W, a.W2, a.lda, a.M, a.N, a.K, a.rows, a.epilogue, a.bias, a.bias_dtype, a.out, a.out_dtype, a.ldo, nm);
  JLLM_CHECK_LAUNCH("gemm_skinny");
  return 0;
}

template <int NW, bool GATED, int WAVES, int PER_CU>
static int launch_skinny_rows(const SkinnyArgs& a, const SkinnyNorm& nm, bool turn, hipStream_t stream) {
  if constexpr (!GATED && PER_CU < 3) {
    if (turn) return a.M <= 8 ? launch_skinny<NW, 1, GATED, WAVES, PER_CU, true>(a, nm, stream) : launch_skinny<NW, 2, GATED, WAVES, PER_CU, true>(a, nm, stream);
  }
  return a.M <= 8 ? launch_skinny<NW, 1, GATED, WAVES, PER_CU, false>(a, nm, stream) : launch_skinny<NW, 2, GATED, WAVES, PER_CU, false>(a, nm, stream);
}

template <int NW, bool GATED>
static int launch_skinny_waves(const SkinnyArgs& a, const SkinnyNorm& nm, int per_cu, bool turn, hipStream_t stream) {
  switch (per_cu) {
    case 1: return launch_skinny_rows<NW, GATED, 8, 1>(a, nm, turn, stream);
    case 2: return launch_skinny_rows<NW, GATED, 4, 2>(a, nm, turn, stream);
    default: return launch_skinny_rows<NW, GATED, 4, 3>(a, nm, turn, stream);
  }
}

static int skinny_checked(const void* A, int lda, const void* W, const void* W2, const void* bias, int bias_dtype,
                          void* out, int out_dtype, int ldo, int M, int N, int K, int epilogue, float gate_limit,
                          const SkinnyNorm& nm_in, int rows, hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (M > 16 || (K & 127) || (N & 15) || (lda & 7) || K <= 0 || lda < 0) return 1;
  if (((uintptr_t)A & 15) || ((uintptr_t)W & 15) || (W2 && ((uintptr_t)W2 & 15))) return 1;
  // a lane's place in an operand is a 32-bit byte offset from the workgroup's first row
  if ((unsigned long long)lda >= (1ull << 26) || (unsigned long long)K >= (1ull << 25)) return 1;
  JLLM_TAKE_GATE("gemm_skinny", epilogue, gate_limit, gs);
  SkinnyNorm nm = nm_in;
  nm.gate = gs;
  if (epilogue < 0 || epilogue > 2 || (epilogue == 2) != (W2 != nullptr)) JLLM_FAIL("gemm_skinny: epilogue %d", epilogue);
  if (epilogue == 1 && out_dtype != JLLM_F32) JLLM_FAIL("gemm_skinny: the accumulate epilogue adds into fp32");
  if (ldo < N) JLLM_FAIL("gemm_skinny: ldo %d < N %d", ldo, N);
  if (rows < 1 || rows > (W2 ? 16 : 32)) JLLM_FAIL("gemm_skinny: %d weight rows per workgroup (1 to 32, gated to 16)", rows);
  const int groups = (N + rows - 1) / rows;
  if (nm.emit_rows && (epilogue != 1 || !nm.emit_gain || !nm.emit_partial)) JLLM_FAIL("gemm_skinny: rows for a norm come from the accumulate epilogue, with gain and partial sums");
  if (nm.emit_rows && nm.emit_parts < groups) JLLM_FAIL("gemm_skinny: %d places for the partial sums of %d workgroups", nm.emit_parts, groups);
  if (nm.norm_partial && nm.norm_parts <= 0) JLLM_FAIL("gemm_skinny: %d partial sums", nm.norm_parts);
  if (nm.norm_partial && ((nm.norm_parts & 3) || ((uintptr_t)nm.norm_partial & 15))) return 1;
  const int cus = jllm_compute_units();
  if (cus <= 0) JLLM_FAIL("gemm_skinny: the GPU's compute units could not be read");
  const SkinnyArgs a{(const bf16_t*)A, (const bf16_t*)W, (const bf16_t*)W2, bias, lda, bias_dtype, out_dtype, ldo, M, N, K, epilogue, rows, out};
  // One workgroup of 8 waves per compute unit where there are no more workgroups than those; else two of 4 waves, so that
  // one streams while the other adds up and stores; three, with a shallower ring, where there are more than two of them and K
  // is so short that a wave has no use for a deep one. Two / three at 1, 8 and 16 rows, us: 151,936 x 1,024 60.7 64.2 67.8 /
  // 54.0 58.1 61.3 (53.4 80.2 91.2 from memory into registers), gated 8,960 x 1,536 15.3 16.4 16.6 / 13.5 14.6 15.0; from K =
  // 2,048 on three are the same to 2 % slower (gated 8,192 x 2,048).
  const int per_cu = groups <= cus ? 1 : groups > 2 * cus && K < 2048 ? 3 : 2;
  // Rows of W that lie a multiple of 4 KB apart, and long rows in workgroups of up to 16 of them: the workgroups begin at
  // different blocks. All at one block, they ask the memory for the same piece of every row at once. One / different at 1, 8 and 16 rows, us:
  // 12,288 x 4,096 22.0 23.4 24.0 / 20.7 22.2 22.6, 4,096 x 11,008 23.2 24.0 25.1 / 19.7 20.3 21.4, 8,192 x 8,192 32.0 34.2
  // 35.4 / 27.7 28.2 28.7, 32,768 x 2,048 30.4 32.1 33.0 / 26.9 29.7 29.8, 4,096 x 4,096 8.9 9.5 10.1 / 8.7 9.1 9.7; slower so:
  // 5,120 x 17,408 (20 rows a workgroup) by 9 %, 7,168 x 5,120 (28) by 4 %.
  const bool turn = K % 2048 == 0 || (rows <= 16 && K >= 8192);
  if (W2) return rows <= 8 ? launch_skinny_waves<1, true>(a, nm, per_cu, false, stream) : launch_skinny_waves<2, true>(a, nm, per_cu, false, stream);
  switch ((rows + 7) / 8) {
    case 1: return launch_skinny_waves<1, false>(a, nm, per_cu, turn, stream);
    case 2: return launch_skinny_waves<2, false>(a, nm, per_cu, turn, stream);
    case 3: return launch_skinny_waves<3, false>(a, nm, per_cu, turn, stream);
    default: return launch_skinny_waves<4, false>(a, nm, per_cu, turn, stream);
  }
}

// `rows`: the weight rows a workgroup owns (1 to 32, with the gated epilogue to 16). returns 0 when it ran, 1 when the
// shape is not one it takes (the caller uses another kernel), -1 on errors
extern "C" int jllm_gemm_skinny_bf16(const void* A, int lda, const void* W, const void* W2, const void* bias,
                                     int bias_dtype, void* out, int out_dtype, int ldo, int M, int N, int K,
                                     int epilogue, float gate_limit, int rows, hipStream_t stream) {
  return skinny_checked(A, lda, W, W2, bias, bias_dtype, out, out_dtype, ldo, M, N, K, epilogue, gate_limit, SkinnyNorm{}, rows, stream);
}

// The same with an RMSNorm on either side (see the head of this file). emit_rows [M, N] bf16, emit_gain [N] and
// emit_partial [M][emit_parts] fp32 (a sum per workgroup, zeros behind them) go with the accumulate epilogue; norm_partial
// [M][norm_parts] with any.
extern "C" int jllm_gemm_skinny_norm_bf16(const void* A, int lda, const void* W, const void* W2, const void* bias,
                                          int bias_dtype, void* out, int out_dtype, int ldo, int M, int N, int K,
                                          int epilogue, float gate_limit, int rows, void* emit_rows, const void* emit_gain,
                                          int emit_gain_dtype, float* emit_partial, int emit_parts, const float* norm_partial,
                                          int norm_parts, float norm_eps, hipStream_t stream) {
  SkinnyNorm nm{(bf16_t*)emit_rows, emit_gain, emit_gain_dtype, emit_partial, emit_parts, norm_partial, norm_parts, norm_eps, GateSpec{0, 0.f}};
  return skinny_checked(A, lda, W, W2, bias, bias_dtype, out, out_dtype, ldo, M, N, K, epilogue, gate_limit, nm, rows, stream);
}
