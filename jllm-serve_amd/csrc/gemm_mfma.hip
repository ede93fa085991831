// out[M,N] = A[M,K] * W[N,K]^T in tiles of 64 x 64 to 256 x 128, for products that the large tiles of gemm_pingpong.hip would leave
// most compute units without: bf16 on the matrix cores (v_mfma_f32_16x16x32_bf16, in the order of that kernel, so both give the
// same outputs).
//
// A wave owns RM x CN accumulators of 16 x 16, WGM x WGN waves a tile. K advances in stages of 64 through a ring of NS stages in
// LDS, filled without registers (global_load_lds_dwordx4, whole lines of 128 bytes, eight rows to an instruction, the bank
// swizzle applied on the global side). A stage's fragments are all in registers before its multiplies begin; between these,
// evenly, a wave reads the next stage's fragments (a second set of registers) and asks for its share of the stage that takes the
// place of the one it is multiplying. One barrier a stage.
//
// What binds is the pipe through which a compute unit fills its LDS (32 bytes a clock at best: 1,024 clocks for a stage of 128 x 128,
// whose MFMAs take 512; a stage takes 0.55 to 0.65 us, some 1,350 clocks, with a tile on nearly every compute unit), and where
// there are few stages the launch, the first bytes and the parts of a cut K. The smaller tiles share a compute unit (two of 64 x 128,
// 72 KB each, two of 64 x 64), which hides one's start and end behind the other.
//
// What stood here before (128 x 128 through registers and two LDS buffers, 32 x 32 x 16; below a thousand rows mostly gemm_stream.hip,
// with LDS reads of 144 KB a stage) / this, us inside a graph, products alone: 0.6B shape at 487 rows qkv 12.2 / 8.9, gate/up 16.8 /
// 14.6, 8B qkv at 128 rows 25.7 / 20.5, at 631 50.9 / 41.4, o at 128 20.1 / 15.
// A ring of two stages (64 KB, four waves) lets two workgroups of 128 x 128 share a compute unit, each stage's loads landing within the stage
// before: the grouped form's, and the per-head form's where it takes many.
//
// Epilogues as in gemm_epilogue.h; K cut over gridDim.z leaves fp32 partial tiles that the reduction below adds up. Two further
// forms: grouped (a workgroup's rows belong to one group, with weights of its own, gathered by an index list) and per head.
// Needs K % 64 == 0 and 16-byte aligned rows; any M and N. The caller falls back otherwise.
#include <type_traits>
#include "common.h"
#include "layer_launches.h"
#include "lds_ring.h"
#include "gemm_epilogue.h"
#include "mfma.h"

#define TBK 64
#define T_ROW_BYTES (TBK * 2)  // a tile row in LDS: 128 bytes = 8 pieces of 16
#define T_FENCE() __builtin_amdgcn_sched_barrier(0)

enum { FORM_PLAIN = 0, FORM_GROUPED = 1, FORM_HEADS = 2, FORM_BY_COLUMNS = 3, FORM_FAR = 4 };  // the last two: plain, in another order of the tiles; of rows of any length

// What the per-head form takes beside the operands: head h = blockIdx.z multiplies the rows at A + h * a_stride with
// its own weights (W [heads][N][K]) and writes bf16 at out + h * o_stride, times sigmoid(gate[row][h * N + column]) where a
// gate is given.
struct HeadsArgs {
  int a_stride, o_stride;
  const bf16_t* gate;
  int ld_gate;
};
// The grouped form: (group, first row, rows) per blockIdx.y, rows = 0 for an unused entry: the workgroup's rows are first ..
// first + rows - 1, its weights those of its group ([groups][N][K]); with `row_map` input row i is row row_map[i] / row_div of A,
// the output rows stay i.
struct GroupArgs {
  const int *groups, *row_map;
  int row_div;
};

// Workgroups go to the eight dies in turn, so with a multiple of eight columns those that share a weight tile are on one die and with
// four more on two; with an odd number every die fetches every weight tile. There workgroups b, b + 8, b + 16 .. (one die) take a
// run of neighbouring tiles, column by column (`by_rows`: 2^32 / rows rounded up; a division would cost 0.3 us). us, by number / so:
// 400 rows of 3,392 x 2,048 in tiles of 64 x 64 (53 columns) 20.4 / 14.1, 1,100 in 64 x 128 (27) 36.6 / 22.5, 1,025 of 6,208 x 4,096 in
// 128 x 256 (25) 74.1 / 54.4, 900 of 22,592 x 4,096 (89) 234.8 / 168.3; ten columns (2,560 x 9,728, 400 rows) 51.4 / 46.2.
// Where the number is a multiple of four it gains nothing (2,560 x 4,096, K whole, in 20 columns of 128: 6 % slower).
static bool by_columns(int rows, int cols) { return rows > 1 && cols % 4 != 0 && (unsigned long long)rows * rows * cols < (1ull << 32); }
static uint32_t by_rows_of(uint32_t rows) { return (uint32_t)(((1ull << 32) + rows - 1) / rows); }
__host__ __device__ __forceinline__ void column_tile(uint32_t b, uint32_t rows, uint32_t cols, uint32_t by_rows, int& row, int& col) {
  const uint32_t tiles = rows * cols, each = tiles >> 3, more = tiles & 7, die = b & 7;
  const uint32_t i = die * each + (die < more ? die : more) + (b >> 3);
  col = (int)(((uint64_t)i * by_rows) >> 32);
  row = (int)(i - col * rows);
}

template <bool GATED, int FORM, int RM, int CN, int WGM, int WGN, int NS>
__global__ __launch_bounds__(WGM* WGN * 64) void gemm_mfma_kernel(
    const bf16_t* __restrict__ A, int lda, const bf16_t* __restrict__ W, const bf16_t* __restrict__ W2,
    const void* __restrict__ bias, int bias_dtype, void* __restrict__ out, int out_dtype, int ldo, int M, int N, int K,
    int epilogue, GateSpec gs, float* __restrict__ partial, GroupArgs ga, HeadsArgs ha, uint32_t by_rows) {
  constexpr int WAVES = WGM * WGN, TBM = WGM * RM * 16, TBN = WGN * CN * 16, STAGE = (TBM + TBN) * T_ROW_BYTES;
  constexpr int LA = TBM / 8 / WAVES, L = LA + TBN / 8 / WAVES;  // load instructions (8 rows each) per wave and stage
  constexpr int NM = 2 * RM * CN, NR = 2 * (RM + CN);            // multiplies and LDS reads of a stage
  // Loads are asked for evenly between the multiplies; with a ring of two stages, where they have to land within this one, at once (4,096
  // rows through 32 experts 199 -> 191 us, 64 experts 800 -> 776)
  constexpr int EVERY = NS == 2 ? 1 : NM / L;
  static_assert(LA * 8 * WAVES == TBM && (L - LA) * 8 * WAVES == TBN && EVERY >= 1, "every wave loads as many rows of either operand");
  static_assert(NS >= 2 && NS <= 6, "one stage being read, the others on their way");
  extern __shared__ __align__(1024) unsigned char smem[];
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int wm = wave / WGN, wn = wave % WGN;
  int row = blockIdx.y, col = blockIdx.x;
  if (FORM == FORM_BY_COLUMNS) column_tile(blockIdx.x + blockIdx.y * gridDim.x, gridDim.y, gridDim.x, by_rows, row, col);
  int m0 = row * TBM;
  if (FORM == FORM_GROUPED) {
    const int rows = ga.groups[3 * row + 2];
    if (rows == 0) return;
    m0 = ga.groups[3 * row + 1];
    M = m0 + rows;
    const size_t at = (size_t)ga.groups[3 * row] * N * K;
    W += at;
    if (GATED) W2 += at;
  }
  if (FORM == FORM_HEADS) {
    A += (size_t)blockIdx.z * ha.a_stride;
    W += (size_t)blockIdx.z * N * K;
  }
  const int n0 = col * (GATED ? TBN / 2 : TBN);  // output columns covered by this workgroup start here
  // gridDim.z > 1: this workgroup multiplies only its share of K and leaves an fp32 partial tile
  const int nk_all = K / TBK;
  const int nk_per = FORM == FORM_HEADS ? nk_all : (nk_all + gridDim.z - 1) / gridDim.z;
  const int kt0 = FORM == FORM_HEADS ? 0 : blockIdx.z * nk_per;
  const int nk = max(0, min(nk_all, kt0 + nk_per) - kt0);

  // ---- global side of the loads: the tile's start at its first stage (the same in all lanes, advanced by scalar arithmetic) and a
  // 32-bit byte offset per lane that never changes (row of the tile and piece: checked on the host). Rows gathered by a list, and those
  // too long for that, lie anywhere: an address per lane.
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)smem;
  const unsigned char* abase = (const unsigned char*)(A + (size_t)m0 * lda) + (size_t)kt0 * T_ROW_BYTES;
  const unsigned char* wbase[2] = {(const unsigned char*)(W + (size_t)n0 * K) + (size_t)kt0 * T_ROW_BYTES,
                                   (const unsigned char*)((GATED ? W2 : W) + (size_t)n0 * K) + (size_t)kt0 * T_ROW_BYTES};
  const unsigned char *base[L], *at[L];
  uint32_t off[L];
#pragma unroll
  for (int c = 0; c < L; ++c) {
    const int chunk = c < LA ? wave * LA + c : wave * (L - LA) + c - LA, r = chunk * 8 + (lane >> 3);
    const uint32_t piece = (uint32_t)(((lane & 7) ^ ring_swz(r)) * 16);
    if (c < LA) {
      const int m = min(r, M - 1 - m0);
      base[c] = abase;
      off[c] = (uint32_t)m * (uint32_t)lda * 2u + piece;
      if (FORM == FORM_GROUPED) {
        const int from = ga.row_map ? ga.row_map[m0 + m] / ga.row_div : m0 + m;
        at[c] = (const unsigned char*)(A + (size_t)from * lda) + piece;
      }
      if (FORM == FORM_FAR) at[c] = base[c] + (size_t)m * lda * 2 + piece;
    } else {  // gated: of a wave's CN blocks of 16 the first half is gate rows, the second the up rows of the same outputs
      const int block = chunk % (2 * CN) / 2;  // the same in all lanes
      const int n = GATED ? chunk / (2 * CN) * CN * 8 + block % (CN / 2) * 16 + (r & 15) : r;
      base[c] = wbase[GATED && block >= CN / 2];
      off[c] = (uint32_t)min(n, N - 1 - n0) * (uint32_t)K * 2u + piece;
      if (FORM == FORM_FAR) at[c] = base[c] + (size_t)min(n, N - 1 - n0) * K * 2 + piece;
    }
  }
  auto load = [&](int t, uint32_t slot, int c) {  // the wave's load c of stage t into the slot at byte `slot`
    const size_t kbytes = (size_t)t * T_ROW_BYTES;
    const uint32_t to = lds0 + slot + (c < LA ? (wave * LA + c) * 1024 : TBM * T_ROW_BYTES + (wave * (L - LA) + c - LA) * 1024);
    if (FORM == FORM_FAR || (FORM == FORM_GROUPED && c < LA))
      load_to_lds_16(at[c] + kbytes, to);
    else
      load_to_lds_16(base[c] + kbytes, off[c], to);
  };
  auto landed = [&](int left) {  // until at most `left` stages of the wave's loads are on their way
    if (NS >= 6 && left >= 4) wait_loads<4 * L>();
    else if (NS >= 5 && left >= 3) wait_loads<3 * L>();
    else if (NS >= 4 && left >= 2) wait_loads<2 * L>();
    else if (left >= 1) wait_loads<L>();
    else wait_loads<0>();
  };
  auto meet = [&] {  // behind the wave's own reads: the stage that it has in registers now is free for the loads of all
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    T_FENCE();
    __builtin_amdgcn_s_barrier();
    T_FENCE();
  };

  // ---- LDS side: fragment of a block of 16 rows: row = block * 16 + lane % 16, piece = lane / 16 (16 bytes: 8 of 32 k), + 4 for the
  // stage's second 32 (bit 6 of the address); 16 rows further leaves ring_swz unchanged
  const int ra = wm * RM * 16 + (lane & 15), rb = wn * CN * 16 + (lane & 15);
  const int aread = ra * T_ROW_BYTES + (((lane >> 4) ^ ring_swz(ra)) * 16);
  const int bread = TBM * T_ROW_BYTES + rb * T_ROW_BYTES + (((lane >> 4) ^ ring_swz(rb)) * 16);
  u32x4 fa[2][2][RM], fb[2][2][CN];  // [set][32 of k][block]
  auto read = [&](int set, uint32_t slot, int x) {  // read x of a stage, in the order of use
    const int kk = x / (RM + CN), y = x % (RM + CN);
    if (y < CN) fb[set][kk][y] = *(const u32x4*)(smem + slot + (bread ^ (kk * 64)) + y * 16 * T_ROW_BYTES);
    else fa[set][kk][y - CN] = *(const u32x4*)(smem + slot + (aread ^ (kk * 64)) + (y - CN) * 16 * T_ROW_BYTES);
  };
  floatx4 acc[RM][CN];
#pragma unroll
  for (int i = 0; i < RM; ++i)
#pragma unroll
    for (int j = 0; j < CN; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};

  // ---- prologue: every stage of the ring on its way, the first in registers, the second landed
#pragma unroll
  for (int s = 0; s < NS; ++s)
    if (s < nk) {
#pragma unroll
      for (int c = 0; c < L; ++c) load(s, s * STAGE, c);
    }
  if (nk >= NS) wait_loads<(NS - 1) * L>();
  else wait_loads<0>();
  meet();
#pragma unroll
  for (int x = 0; x < NR; ++x) read(0, 0, x);
  if (nk >= NS) wait_loads<(NS - 2) * L>();
  meet();
  // Stage t is multiplied from one set of registers while stage t + 1 (its slot: rs) is read into the other and stage t + NS loaded into
  // the slot of stage t (ws). At its end stage t + 2 has landed: each wave waits for its own loads, the barrier for all waves.
  uint32_t rs = STAGE, ws = 0;
  auto stage = [&](auto which, auto full, int t) {
    constexpr int SET = decltype(which)::value;
    constexpr bool FULL = decltype(full)::value;  // not among the last stages: every load is asked for
    const int p = t + NS;
#pragma unroll
    for (int n = 0; n < NM; ++n) {
      const int kk = n / (RM * CN), i = n % (RM * CN) / CN, j = n % CN;
      // the weight fragment goes in as the first operand: the accumulator then holds the tile transposed (rows = output
      // columns), so a lane owns four consecutive output columns of one row and stores them at once
      acc[i][j] = mfma16(fb[SET][kk][j], fa[SET][kk][i], acc[i][j]);
      T_FENCE();
      if (n < NR) {
        read(1 - SET, rs, n);
        T_FENCE();
      }
      if (n == NM - 1) {
#pragma unroll
        for (int x = NM; x < NR; ++x) read(1 - SET, rs, x);
      }
      if (n % EVERY == EVERY / 2 && n / EVERY < L && (FULL || p < nk)) {
        load(p, ws, n / EVERY);
        T_FENCE();
      }
    }
    landed(FULL ? NS - 2 : min(p, nk - 1) - (t + 2));
    meet();
    rs = rs == (NS - 1) * STAGE ? 0 : rs + STAGE;
    ws = ws == (NS - 1) * STAGE ? 0 : ws + STAGE;
  };
  int t = 0;
  for (; t + 1 < nk - NS; t += 2) {
    stage(std::integral_constant<int, 0>{}, std::true_type{}, t);
    stage(std::integral_constant<int, 1>{}, std::true_type{}, t + 1);
  }
  for (; t < nk; t += 2) {  // (the reads behind the last stage fetch some slot's bytes, which are never multiplied)
    stage(std::integral_constant<int, 0>{}, std::false_type{}, t);
    if (t + 1 < nk) stage(std::integral_constant<int, 1>{}, std::false_type{}, t + 1);
  }
  if (FORM == FORM_HEADS) {
    bf16_t* o = (bf16_t*)out + (size_t)blockIdx.z * ha.o_stride;
#pragma unroll
    for (int i = 0; i < RM; ++i) {
      const int m = m0 + (wm * RM + i) * 16 + (lane & 15);
      if (m >= M) continue;
#pragma unroll
      for (int j = 0; j < CN; ++j) {
        const int n = n0 + (wn * CN + j) * 16 + (lane >> 4) * 4;
        if (n >= N) continue;  // N is a multiple of four
        floatx4 v = acc[i][j];
        if (ha.gate) {
          const u32x2 g = *(const u32x2*)(ha.gate + (size_t)m * ha.ld_gate + (size_t)blockIdx.z * N + n);
          const float gv[4] = {__uint_as_float(g[0] << 16), __uint_as_float(g[0] & 0xffff0000u), __uint_as_float(g[1] << 16),
                               __uint_as_float(g[1] & 0xffff0000u)};
#pragma unroll
          for (int c = 0; c < 4; ++c) v[c] = v[c] / (1.0f + __expf(-gv[c]));
        }
        *(u32x2*)(o + (size_t)m * ldo + n) = u32x2{pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3])};
      }
    }
    return;
  }
  tile_epilogue<GATED, RM, CN, TBM, TBN>(acc, lane, wm, wn, m0, n0, bias, bias_dtype, out, out_dtype, ldo, M, N, epilogue, gs, partial,
                                             (int)blockIdx.z, (int)gridDim.z);
}

// sums the K-split partials in ascending order of the split and applies bias and epilogue; V outputs per thread
// (4 when the rows allow 16-byte accesses)
template <int V>
__global__ __launch_bounds__(256) void splitk_reduce_kernel(const float* __restrict__ partial, int splits,
                                                            const void* __restrict__ bias, int bias_dtype,
                                                            void* __restrict__ out, int out_dtype, int ldo, int M, int N,
                                                            int epilogue) {
  const size_t i = ((size_t)blockIdx.x * 256 + threadIdx.x) * V;
  if (i >= (size_t)M * N) return;
  const int m = (int)(i / N), n = (int)(i % N);
  float v[V];
#pragma unroll
  for (int e = 0; e < V; ++e) v[e] = 0.f;
  for (int z = 0; z < splits; ++z) {
    const float* p = partial + (size_t)z * M * N + i;
    if (V == 4) {
      const float4 t = *(const float4*)p;
      v[0] += t.x, v[1 % V] += t.y, v[2 % V] += t.z, v[3 % V] += t.w;
    } else {
      v[0] += p[0];
    }
  }
  if (bias) {
#pragma unroll
    for (int e = 0; e < V; ++e)
      v[e] += (bias_dtype == JLLM_BF16) ? ldf((const bf16_t*)bias, n + e) : ldf((const float*)bias, n + e);
  }
  const size_t o = (size_t)m * ldo + n;
  if (epilogue == 1) {
    float* r = (float*)out + o;
    if (V == 4) {
      float4 t = *(float4*)r;
      t.x += v[0], t.y += v[1 % V], t.z += v[2 % V], t.w += v[3 % V];
      *(float4*)r = t;
    } else {
      r[0] += v[0];
    }
  } else if (out_dtype == JLLM_BF16) {
#pragma unroll
    for (int e = 0; e < V; ++e) stf((bf16_t*)out, o + e, v[e]);
  } else {
#pragma unroll
    for (int e = 0; e < V; ++e) stf((float*)out, o + e, v[e]);
  }
}

// The reduction of a product that adds into the residual, and the RMSNorm of the new rows, in one pass: a workgroup per row,
// which stays in registers (N <= 8,192, a multiple of 4, rows without gaps), everything it reads requested before the first
// sum. The bits are those of the reduction above followed by the norm kernel (elementwise.hip): parts in ascending order, bias,
// residual, then the squares by thread, wave and block. Bound by its bytes; the norm's own pass read the rows again
// and cost a launch: 2,048 rows of 4,096 in two parts 22.4 + 13.4 -> 25.7 us, 631 in four 10.1 + 6.6 -> 12.5. (With a branch
// around every load, as in the kernels it replaces, 46 and 22.)
template <typename TG, int J>
__global__ __launch_bounds__(256) void splitk_reduce_norm_kernel(const float* __restrict__ partial, int splits, const void* __restrict__ bias,
                                                                 int bias_dtype, float* __restrict__ out, int M, int N,
                                                                 const TG* __restrict__ gain, float eps, bf16_t* __restrict__ rows, int ldr) {
  __shared__ float red[4];
  const int nv = N >> 2;  // fours of a row: thread t has number t, t + 256, ..; beyond the end it reads the last one again (no
                          // branch around a load: the compiler would wait for everything behind one)
  const size_t row = (size_t)blockIdx.x * N;
  int at[J];
  floatx4 v[J], res[J];
  TG g[J][4];
#pragma unroll
  for (int j = 0; j < J; ++j) {
    at[j] = 4 * min((int)threadIdx.x + 256 * j, nv - 1);
    v[j] = floatx4{0.f, 0.f, 0.f, 0.f};
    res[j] = *(const floatx4*)(out + row + at[j]);
    if (sizeof(TG) == 2)
      *(uint2*)g[j] = *(const uint2*)(gain + at[j]);
    else
      *(uint4*)g[j] = *(const uint4*)(gain + at[j]);
  }
  int z = 0;
  for (; z + 2 <= splits; z += 2) {
    const float* p = partial + (size_t)z * M * N + row;
    const float* p2 = p + (size_t)M * N;
    floatx4 a[J], b[J];
#pragma unroll
    for (int j = 0; j < J; ++j) a[j] = *(const floatx4*)(p + at[j]);
#pragma unroll
    for (int j = 0; j < J; ++j) b[j] = *(const floatx4*)(p2 + at[j]);
#pragma unroll
    for (int j = 0; j < J; ++j) v[j] = (v[j] + a[j]) + b[j];
  }
  if (z < splits) {
#pragma unroll
    for (int j = 0; j < J; ++j) v[j] += *(const floatx4*)(partial + (size_t)z * M * N + row + at[j]);
  }
  float ss = 0.f;
#pragma unroll
  for (int j = 0; j < J; ++j) {
    if (bias)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        v[j][e] += (bias_dtype == JLLM_BF16) ? ldf((const bf16_t*)bias, at[j] + e) : ldf((const float*)bias, at[j] + e);
    v[j] = res[j] + v[j];
    if ((int)threadIdx.x + 256 * j < nv) {
      *(floatx4*)(out + row + at[j]) = v[j];
      ss += v[j][0] * v[j][0] + v[j][1] * v[j][1] + v[j][2] * v[j][2] + v[j][3] * v[j][3];
    }
  }
  ss = block_sum<4>(ss, red);
  const float s = norm_scale(ss, N, eps);
  bf16_t* o = rows + (size_t)blockIdx.x * ldr;
#pragma unroll
  for (int j = 0; j < J; ++j) {
    if ((int)threadIdx.x + 256 * j >= nv) continue;
    float r[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) r[e] = (v[j][e] * s) * ldf(g[j], e);
    *(uint2*)(o + at[j]) = uint2{(uint32_t)f32_to_bf16(r[0]).bits | ((uint32_t)f32_to_bf16(r[1]).bits << 16),
                                 (uint32_t)f32_to_bf16(r[2]).bits | ((uint32_t)f32_to_bf16(r[3]).bits << 16)};
  }
}

int jllm_splitk_reduce_norm(const float* partial, int splits, const void* bias, int bias_dtype, void* out, int out_dtype, int ldo, int M, int N,
                            int epilogue, const void* gain, int gain_dtype, float eps, void* rows, int ldr, hipStream_t stream) {
  if (epilogue != 1 || out_dtype != JLLM_F32 || ldo != N || (N & 3) || N > 8192 || ldr < N || (ldr & 3) || !gain || (((uintptr_t)out | (uintptr_t)partial) & 15) ||
      ((uintptr_t)rows & 7))
    JLLM_FAIL("splitk_reduce_norm: rows of %d (stride %d) and a norm's of stride %d", N, ldo, ldr);
  if ((uintptr_t)gain & 15) JLLM_FAIL("splitk_reduce_norm: a gain that is not aligned to 16 bytes");
#define SRN_CASE(J)                                                                                                                                    \
  case J:                                                                                                                                              \
    splitk_reduce_norm_kernel<TG, J><<<M, 256, 0, stream>>>(partial, splits, bias, bias_dtype, (float*)out, M, N, (const TG*)gain, eps, (bf16_t*)rows, ldr); \
    break;
  JLLM_DISPATCH_1(gain_dtype, TG, {
    switch ((N / 4 + 255) / 256) {
      SRN_CASE(1) SRN_CASE(2) SRN_CASE(3) SRN_CASE(4) SRN_CASE(5) SRN_CASE(6) SRN_CASE(7) SRN_CASE(8)
    }
  })
#undef SRN_CASE
  JLLM_CHECK_LAUNCH("splitk_reduce_norm");
  return 0;
}

int jllm_splitk_reduce(const float* partial, int splits, const void* bias, int bias_dtype, void* out, int out_dtype,
                       int ldo, int M, int N, int epilogue, hipStream_t stream) {
  const size_t total = (size_t)M * N;
  if ((N & 3) == 0 && (ldo & 3) == 0 && ((uintptr_t)out & 15) == 0 && ((uintptr_t)partial & 15) == 0) {
    splitk_reduce_kernel<4><<<(unsigned)((total / 4 + 255) / 256), 256, 0, stream>>>(partial, splits, bias, bias_dtype, out,
                                                                                   out_dtype, ldo, M, N, epilogue);
  } else {
    splitk_reduce_kernel<1><<<(unsigned)((total + 255) / 256), 256, 0, stream>>>(partial, splits, bias, bias_dtype, out,
                                                                               out_dtype, ldo, M, N, epilogue);
  }
  JLLM_CHECK_LAUNCH("splitk_reduce");
  return 0;
}

// For tests: the row and column (out[0], out[1]) of the tile that workgroup b of a plain product's rows x cols takes
extern "C" int jllm_tiled_place(int rows, int cols, int b, int* out) {
  if (rows < 1 || cols < 1 || b < 0 || b >= rows * cols) return -1;
  out[0] = b / cols, out[1] = b % cols;
  if (by_columns(rows, cols)) column_tile(b, rows, cols, by_rows_of(rows), out[0], out[1]);
  return 0;
}

// the kernel of a tile, its dynamic LDS allowed for
template <bool GATED, int FORM, int RM, int CN, int WGM, int WGN, int NS>
struct Tiled {
  static constexpr int ROWS = WGM * RM * 16, COLS = WGN * CN * 16 / (GATED ? 2 : 1), THREADS = WGM * WGN * 64;
  static constexpr int LDS = (WGM * RM * 16 + WGN * CN * 16) * T_ROW_BYTES * NS;
  static_assert(LDS <= 160 * 1024, "the ring fits");
  static bool allow() {
    static bool allowed = false;
    if (!allowed)
      allowed = hipFuncSetAttribute((const void*)gemm_mfma_kernel<GATED, FORM, RM, CN, WGM, WGN, NS>, hipFuncAttributeMaxDynamicSharedMemorySize, LDS) == hipSuccess;
    return allowed;
  }
};

template <bool GATED, int FORM, int RM, int CN, int WGM, int WGN, int NS>
static int launch_tiled_as(dim3 grid, uint32_t by_rows, const void* A, int lda, const void* W, const void* W2, const void* bias, int bias_dtype,
                           void* out, int out_dtype, int ldo, int M, int N, int K, int epilogue, GateSpec gs, float* partial, hipStream_t stream) {
  using T = Tiled<GATED, FORM, RM, CN, WGM, WGN, NS>;
  if (!T::allow()) JLLM_FAIL("gemm_mfma: cannot reserve %d bytes of LDS", T::LDS);
  gemm_mfma_kernel<GATED, FORM, RM, CN, WGM, WGN, NS><<<grid, T::THREADS, T::LDS, stream>>>(
      (const bf16_t*)A, lda, (const bf16_t*)W, (const bf16_t*)W2, bias, bias_dtype, out, out_dtype, ldo, M, N, K, epilogue, gs, partial, GroupArgs{}, HeadsArgs{}, by_rows);
  return 0;
}

template <bool GATED, int RM, int CN, int WGM, int WGN, int NS, bool FAR = false>
static int launch_tiled(const void* A, int lda, const void* W, const void* W2, const void* bias, int bias_dtype,
                        void* out, int out_dtype, int ldo, int M, int N, int K, int epilogue, GateSpec gs, int splits,
                        float* partial, hipStream_t stream) {
  using T = Tiled<GATED, FORM_PLAIN, RM, CN, WGM, WGN, NS>;
  const dim3 grid((N + T::COLS - 1) / T::COLS, (M + T::ROWS - 1) / T::ROWS, splits);
  if (grid.y > 65535) return 1;
  if constexpr (FAR)
    return launch_tiled_as<GATED, FORM_FAR, RM, CN, WGM, WGN, NS>(grid, 0, A, lda, W, W2, bias, bias_dtype, out, out_dtype, ldo, M, N, K, epilogue, gs, partial, stream);
  if (by_columns(grid.y, grid.x))
    return launch_tiled_as<GATED, FORM_BY_COLUMNS, RM, CN, WGM, WGN, NS>(grid, by_rows_of(grid.y), A, lda, W, W2, bias, bias_dtype, out, out_dtype, ldo, M, N, K, epilogue, gs, partial, stream);
  return launch_tiled_as<GATED, FORM_PLAIN, RM, CN, WGM, WGN, NS>(grid, 0, A, lda, W, W2, bias, bias_dtype, out, out_dtype, ldo, M, N, K, epilogue, gs, partial, stream);
}

// a tile's rows of either operand, of which there are at most so many, lie within 32-bit byte offsets
static bool tiled_rows_fit(int a_rows, int lda, int w_rows, int K) { return (uint64_t)a_rows * lda * 2 < (1ull << 32) && (uint64_t)w_rows * K * 2 < (1ull << 32); }

// `tile`: rows * 1000 + columns of the output tile (of both products' columns with the gated epilogue): 64064 (not gated), 64128, 128128,
// 128256, 256128.
// `splits` > 1 cuts K over gridDim.z (not with the gated epilogue; any count that leaves no part without); `partial` then holds
// splits * M * N floats.
// `norm_rows` [M][norm_ld] bf16 (with cuts of K and the accumulate epilogue): the RMSNorm of the new rows, made by the reduction.
// Rows of 16 MB and more go through tiles of 128 x 128 with an address per lane, whatever the tile.
// returns 0 when it ran, 1 when the shape is not one it takes, -1 on errors
extern "C" int jllm_gemm_mfma_bf16(const void* A, int lda, const void* W, const void* W2, const void* bias,
                                   int bias_dtype, void* out, int out_dtype, int ldo, int M, int N, int K, int epilogue,
                                   float gate_limit, int tile, int splits, float* partial, const void* norm_gain, int norm_gain_dtype, float norm_eps,
                                   void* norm_rows, int norm_ld, hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (K <= 0 || (K % TBK) || (lda & 7)) return 1;
  if (((uintptr_t)A & 15) || ((uintptr_t)W & 15) || (W2 && ((uintptr_t)W2 & 15))) return 1;
  JLLM_TAKE_GATE("gemm_mfma", epilogue, gate_limit, gs);
  if (epilogue < 0 || epilogue > 2 || (epilogue == 2) != (W2 != nullptr)) JLLM_FAIL("gemm_mfma: epilogue %d", epilogue);
  if (epilogue == 1 && out_dtype != JLLM_F32) JLLM_FAIL("gemm_mfma: the accumulate epilogue adds into fp32");
  if (ldo < N) JLLM_FAIL("gemm_mfma: ldo %d < N %d", ldo, N);
  if (splits < 1) splits = 1;
  const int stages = K / TBK, per = (stages + splits - 1) / splits;
  if (splits > 1 && (W2 || !partial || splits > 65535 || stages <= per * (splits - 1))) JLLM_FAIL("gemm_mfma: %d K splits are not possible here", splits);
  if (norm_rows && splits == 1) JLLM_FAIL("gemm_mfma: the norm is the reduction's, and K is whole");
  int rc;
#define TILED_CASE(CODE, ...)                                                                                                                       \
  case CODE:                                                                                                                                        \
    rc = W2 ? launch_tiled<true, __VA_ARGS__>(A, lda, W, W2, bias, bias_dtype, out, out_dtype, ldo, M, N, K, epilogue, gs, 1, partial, stream)       \
            : launch_tiled<false, __VA_ARGS__>(A, lda, W, W2, bias, bias_dtype, out, out_dtype, ldo, M, N, K, epilogue, gs, splits, partial, stream); \
    break;
  switch (tiled_rows_fit(256, lda, 256, K) ? tile : -1) {
    TILED_CASE(-1, 2, 4, 4, 2, 5, true)
    TILED_CASE(64128, 2, 4, 2, 2, 3)
    TILED_CASE(128128, 2, 4, 4, 2, 5)
    TILED_CASE(128256, 4, 4, 2, 4, 3)
    TILED_CASE(256128, 4, 4, 4, 2, 3)
    case 64064:
      if (!W2) {
        rc = launch_tiled<false, 2, 2, 2, 2, 4>(A, lda, W, W2, bias, bias_dtype, out, out_dtype, ldo, M, N, K, epilogue, gs, splits, partial, stream);
        break;
      }
      [[fallthrough]];
    default:
      JLLM_FAIL("gemm_mfma: no tile of %d rows x %d columns here", tile / 1000, tile % 1000);
  }
#undef TILED_CASE
  if (rc != 0) return rc;
  JLLM_CHECK_LAUNCH("gemm_mfma");
  if (splits > 1 && norm_rows)
    return jllm_splitk_reduce_norm(partial, splits, bias, bias_dtype, out, out_dtype, ldo, M, N, epilogue, norm_gain, norm_gain_dtype, norm_eps, norm_rows, norm_ld, stream);
  if (splits > 1) return jllm_splitk_reduce(partial, splits, bias, bias_dtype, out, out_dtype, ldo, M, N, epilogue, stream);
  return 0;
}

// The grouped form in tiles of 128 x 128, four waves and a ring of two stages, so that two workgroups share a compute unit: at few rows an
// expert the weights' way from memory is what binds, at many the tiles' starts and ends, and either needs another workgroup beside. us, what
// stood here before the rings / a ring of five stages, one workgroup a compute unit / this (rows x 4 through 32 experts of 1,024 x 2,048,
// x 6 through 64 of 1,536 x 4,096): gate/up of 512 rows 47.8 / 56.7 / 49.6, of 1,024 89.5 / 88.4 / 84.9, of 4,096 222 / 212 / 191 and 877 /
// 857 / 776; down 31.2 / 35.9 / 32.3, 47.8 / 56.3 / 43.5, 128 / 143 / 121 and 514 / 555 / 466. Tiles of 128 x 64 in rings of three: gate/up 59.4,
// 84.6, 224 and 986.
// `tiles` holds (group, first row, rows <= 128) per entry (rows = 0: unused), the
// weights are [groups][N][K] (and W2 likewise for the gated epilogue), row i of the input is A[row_map[i] / row_div]
// when `row_map` is given, and output row i is row i of `out`. K whole, epilogues store and gated.
// returns 0 when it ran, 1 when the shape is not one it takes, -1 on errors
extern "C" int jllm_gemm_mfma_grouped_bf16(const void* A, int lda, const void* W, const void* W2, void* out, int out_dtype,
                                           int ldo, int M, int N, int K, int epilogue, float gate_limit, const int* tiles,
                                           int max_tiles, int tile_rows, const int* row_map, int row_div,
                                           hipStream_t stream) {
  if (max_tiles <= 0 || M <= 0) return 0;
  if ((K & 63) || K <= 0 || N <= 0 || (lda & 7) || max_tiles > 65535 || !tiled_rows_fit(0, lda, 128, K)) return 1;
  if (((uintptr_t)A & 15) || ((uintptr_t)W & 15) || (W2 && ((uintptr_t)W2 & 15))) return 1;
  JLLM_TAKE_GATE("gemm_mfma_grouped", epilogue, gate_limit, gs);
  if ((epilogue != 0 && epilogue != 2) || (epilogue == 2) != (W2 != nullptr)) JLLM_FAIL("gemm_mfma_grouped: epilogue %d", epilogue);
  using Plain = Tiled<false, FORM_GROUPED, 4, 4, 2, 2, 2>;
  using Gated = Tiled<true, FORM_GROUPED, 4, 4, 2, 2, 2>;
  if (tile_rows != Plain::ROWS) JLLM_FAIL("gemm_mfma_grouped: tiles of %d rows, this kernel takes %d", tile_rows, Plain::ROWS);
  if (ldo < N || row_div < 1) JLLM_FAIL("gemm_mfma_grouped: ldo %d < N %d", ldo, N);
  const int cols = W2 ? Gated::COLS : Plain::COLS;
  dim3 grid((N + cols - 1) / cols, max_tiles, 1);
  if (!Plain::allow() || !Gated::allow()) JLLM_FAIL("gemm_mfma_grouped: cannot reserve %d bytes of LDS", Plain::LDS);
  const GroupArgs ga{tiles, row_map, row_div};
  if (W2)
    gemm_mfma_kernel<true, FORM_GROUPED, 4, 4, 2, 2, 2><<<grid, Gated::THREADS, Gated::LDS, stream>>>(
        (const bf16_t*)A, lda, (const bf16_t*)W, (const bf16_t*)W2, nullptr, 0, out, out_dtype, ldo, M, N, K, epilogue, gs, nullptr, ga, HeadsArgs{}, 0);
  else
    gemm_mfma_kernel<false, FORM_GROUPED, 4, 4, 2, 2, 2><<<grid, Plain::THREADS, Plain::LDS, stream>>>(
        (const bf16_t*)A, lda, (const bf16_t*)W, nullptr, nullptr, 0, out, out_dtype, ldo, M, N, K, epilogue, gs, nullptr, ga, HeadsArgs{}, 0);
  JLLM_CHECK_LAUNCH("gemm_mfma_grouped");
  return 0;
}

template <int RM, int CN, int WGM, int WGN, int NS>
static int launch_heads(const void* in, int ld_in, int in_hstride, const void* W, void* out, int ld_out, int out_hstride, int M,
                        int H, int N, int K, const void* gate, int ld_gate, hipStream_t stream) {
  using T = Tiled<false, FORM_HEADS, RM, CN, WGM, WGN, NS>;
  if (!tiled_rows_fit(T::ROWS, ld_in, T::COLS, K)) return 1;
  dim3 grid((N + T::COLS - 1) / T::COLS, (M + T::ROWS - 1) / T::ROWS, H);
  if (grid.y > 65535) return 1;
  if (!T::allow()) JLLM_FAIL("gemm_mfma_heads: cannot reserve %d bytes of LDS", T::LDS);
  gemm_mfma_kernel<false, FORM_HEADS, RM, CN, WGM, WGN, NS><<<grid, T::THREADS, T::LDS, stream>>>(
      (const bf16_t*)in, ld_in, (const bf16_t*)W, nullptr, nullptr, 0, out, JLLM_BF16, ld_out, M, N, K, 0, GateSpec{}, nullptr, GroupArgs{},
      HeadsArgs{in_hstride, out_hstride, (const bf16_t*)gate, ld_gate}, 0);
  JLLM_CHECK_LAUNCH("gemm_mfma_heads");
  return 0;
}

// The per-head products of latent attention for many rows (latent_heads.hip, which checks the arguments): K a multiple of
// 64, N of 4. Through LDS a row's and a weight's loads are shared by a workgroup, two of which share a compute unit: tiles of 64 x 128 in
// rings of three stages, or of 128 x 128 in rings of two where these take fewer rounds of workgroups (a round of one to a compute unit
// 0.6 of one of two; one of 128 x 128 1.66 of 64 x 128). us, straight from memory by every wave (64 x 64 outputs each) / 64 x 128 / 128 x
// 128, 512 x 128: 16 heads at 500 rows 11.9 / 7.4 / 7.5, at 2,556 42.2 / 24.9 / 24.0, 64 heads at 65 rows - / 8.2 / 6.7, 32 heads at 2,556
// - / 55.2 / 41.9; 128 x 512 with a gate: 16 heads at 65 rows 14.4 / 8.6 / 11.9, at 2,556 41 / 21.2 / 22.3, 64 heads at 800 - / 29.0 / 28.0.
int jllm_gemm_mfma_heads(const void* in, int ld_in, int in_hstride, const void* W, void* out, int ld_out, int out_hstride, int M,
                         int H, int N, int K, const void* gate, int ld_gate, hipStream_t stream) {
  const long cus = jllm_compute_units(), cols = (N + 127) / 128;
  auto rounds = [&](int rows) {  // of two workgroups to a compute unit
    const long groups = ((M + rows - 1) / rows) * cols * H, last = groups % (2 * cus);
    return groups / (2 * cus) + (last == 0 ? 0.0 : last <= cus ? 0.6 : 1.0);
  };
  if (rounds(64) < 1.66 * rounds(128))
    return launch_heads<2, 4, 2, 2, 3>(in, ld_in, in_hstride, W, out, ld_out, out_hstride, M, H, N, K, gate, ld_gate, stream);
  return launch_heads<4, 4, 2, 2, 2>(in, ld_in, in_hstride, W, out, ld_out, out_hstride, M, H, N, K, gate, ld_gate, stream);
}
