// out[M,N] = A[M,K] * W[N,K]^T for 17 to 64 rows (decode steps of many requests, small prompt portions), bound by streaming W
// from HBM once, and for the smaller products of up to about a thousand (gridDim.z tiles of 64 or 128 rows): bf16 operands,
// fp32 accumulation on the matrix cores (16x16x32).
//
// A workgroup owns CT tiles of 16 weight rows (gated: half of them gate, half up) and a range of K, with two waves per
// tile: in a block of 64 k one takes the first 32, the other the rest, each for all the activation rows. Both operands go
// straight from memory into a ring of S blocks in LDS (global_load_lds_dwordx4, 8 rows of 128 bytes per instruction,
// bank swizzle applied on the global side), S - 1 blocks ahead of the multiplies; one barrier per block.
//
// What binds a compute unit here is its load pipe, through which the activations go as well (about 39 bytes a nanosecond
// for such loads). So a workgroup should own about as many weight rows as there are activation rows, or more, and where
// that leaves compute units without one, K is cut over gridDim.y. Each part leaves its sums, with accesses that pass the
// caches by (common.h), and the workgroup of a column tile that arrives last adds the parts in ascending order and applies
// bias and epilogue: no second launch. Up to 64 rows, how N and K are cut depends on N and K only, never on M: a row's result
// does not depend on the rows beside it. Beyond, tiles and parts follow M, and with them the order of a row's sums and of the
// squares that a norm adds up.
//
// Inside a graph, us at 20, 32 and 64 rows, before (fragments of the weights straight from memory a step ahead, 128 rows per
// workgroup, the parts added by a second launch) / now: 8B shape qkv 19.4 20.0 22.6 / 16.7 17.3 20.8, o 13.5 14.1 16.7 /
// 12.4 13.1 16.3, gate/up 51.8 53.7 58.6 / 41.9 41.7 43.1, down 28.2 29.1 32.7 / 24.4 25.2 30.3; 0.6B shape qkv 11.6 11.7 13.5 /
// 6.7 6.9 8.4, o 10.2 10.4 11.7 / 7.1 7.4 9.2, gate/up 17.8 18.1 19.8 / 7.5 8.2 9.3, down 11.2 11.4 12.9 / 8.4 8.6 10.7; a step
// of 64 requests of the 8B shape 6.47 -> 5.42 ms. A large copy's rate (6.2 TB/s) would take 8.1, 5.4, 32.5 and 16.2 us of the
// 8B shape's four; the rest is the launch and the first bytes (4), the parts' way through memory (3, 4 and more at 64 rows) and
// at 64 rows the load pipe.
//
// The norm forms are those of the kernel for up to 16 rows: "emit" leaves bf16(new residual * gain) and a sum of squares per
// workgroup for the norm that follows, "normed" multiplies the sums by rsqrt(sum of the input rows' partial sums of squares
// / K + eps).
//
// Needs K % 128 == 0, N % 16 == 0, 16-byte aligned rows; the caller uses another kernel otherwise.
#include "common.h"
#include "layer_launches.h"
#include "lds_ring.h"
#include "mfma.h"

#define GS_ROW_BYTES 128  // a row of a block in LDS: 64 k = 8 pieces of 16 bytes

struct StreamNorm {
  bf16_t* emit_rows;
  int emit_ld;
  const void* emit_gain;
  int emit_gain_dtype;
  float* emit_partial;  // [M][emit_parts]: a sum per column tile, zeros behind them
  int emit_parts;
  const float* norm_partial;
  int norm_parts;
  float norm_eps;
};

struct StreamArgs {
  const bf16_t *A, *W, *W2;
  const void* bias;
  void* out;
  float* partial;  // [column tile][part][tile of 16][tile of 16 rows][lane][4]
  int* arrivals;   // [column tile], zeros, left as zeros
  int lda, bias_dtype, out_dtype, ldo, M, N, K, epilogue, blocks_per_part, turn;
  GateSpec gate;
  StreamNorm nm;
};

// until at most n of the wave's loads are in flight (more than that may have landed)
__device__ __forceinline__ void gs_wait_at_most(int n) {
  switch (n) {
    case 0: return wait_loads<0>();
    case 1: return wait_loads<1>();
    case 2: return wait_loads<2>();
    case 3: return wait_loads<3>();
    case 4: return wait_loads<4>();
    case 5: return wait_loads<5>();
    case 6: return wait_loads<6>();
    case 7: return wait_loads<7>();
    case 8: return wait_loads<8>();
    case 9: return wait_loads<9>();
    case 10: return wait_loads<10>();
    case 11: return wait_loads<11>();
    case 12: return wait_loads<12>();
    case 13: case 14: return wait_loads<13>();
    case 15: case 16: case 17: return wait_loads<15>();
    default: return wait_loads<18>();
  }
}

// a wave's loads per block as a constant: f(GsLoads<n>) for n from 1 to NL
template <int N>
struct GsLoads {
  static constexpr int n = N;
};
template <int NL, typename F>
__device__ __forceinline__ void gs_with_loads(int n, F f) {
  if constexpr (NL > 1) {
    if (n < NL) return gs_with_loads<NL - 1>(n, f);
  }
  f(GsLoads<NL>{});
}

// blocks in the ring: one workgroup per compute unit, or two (`shared`); 3 KB (5 for more rows) stay for what is not the ring
constexpr int gs_slots(int ct, int mt, bool shared) {
  const int fit = ((shared ? 80 : 160) - (mt > 4 ? 5 : 3)) / (2 * ct + 2 * mt);
  return fit > 8 ? 8 : fit;
}

template <int CT, int MT, bool GATED, bool SHARED>
__global__ __launch_bounds__(CT * 128, SHARED ? CT : 1) void gemm_stream_kernel(StreamArgs p) {
  constexpr int NW = 2 * CT;                // waves
  constexpr int BLOCK = (2 * CT + 2 * MT) * 1024;
  constexpr int S = gs_slots(CT, MT, SHARED);
  constexpr int OT = GATED ? CT / 2 : CT;   // tiles of outputs
  constexpr int AL = (2 * MT + NW - 1) / NW;  // activation loads of a wave, at most
  constexpr int MAX_ROWS = MT > 4 ? 128 : 64;
  constexpr int TPR = (CT == 2 ? 4 : 8) * 64 / MAX_ROWS;  // normed: threads that add up a row's squares
  static_assert(S >= 3 && (S - 1) * (1 + AL) < 63 && S * BLOCK >= 2 * CT * MT * 1024, "the ring and what it holds afterwards");
  extern __shared__ __align__(1024) unsigned char smem[];
  __shared__ float rs[MAX_ROWS];            // normed: the rows' scales
  __shared__ float rowsq[OT][MAX_ROWS];     // emit: the squares of a row's columns, per tile
  __shared__ int last;
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int col = lane & 15, g = lane >> 4;
  const int ct = wave >> 1, kg = wave & 1;  // the wave's tile of weight rows and its half of a block
  const int n0 = blockIdx.x * OT * 16;
  const int nblk = p.K >> 6;
  const int b_first = blockIdx.y * p.blocks_per_part;
  const int total = min(nblk - b_first, p.blocks_per_part);
  const int parts = gridDim.y;
  {  // the workgroup's rows
    const int m0 = blockIdx.z * MT * 16;
    p.M = min(p.M - m0, MT * 16);
    p.A += (size_t)m0 * p.lda;
    p.out = p.out_dtype == JLLM_BF16 ? (void*)((bf16_t*)p.out + (size_t)m0 * p.ldo) : (void*)((float*)p.out + (size_t)m0 * p.ldo);
    if (p.nm.norm_partial) p.nm.norm_partial += (size_t)m0 * p.nm.norm_parts;
    if (p.nm.emit_rows) {
      p.nm.emit_rows += (size_t)m0 * p.nm.emit_ld;
      p.nm.emit_partial += (size_t)m0 * p.nm.emit_parts;
    }
  }
  const size_t tile = blockIdx.x + (size_t)gridDim.x * blockIdx.z;
  // up to 64 rows and K whole: column tiles walk K from different blocks, so that workgroups do not all ask the same memory
  // channels at once (rows are often a multiple of 4 KB apart; 8B gate/up at 20 rows 45.5 -> 43.3 us; with parts of K the same
  // or 1 us slower, and for more rows an output's bits would follow the choice of tiles)
  const int rot = p.turn ? (int)((blockIdx.x * 5u) % (unsigned)total) : 0;
  // normed: thread tid % TPR of row tid / TPR adds up the fours of squares number tid % TPR, + TPR, ...; the first two are
  // requested before anything else and added up behind the products
  floatx4 first[2];
  const int sq_row = tid / TPR, sq_at = tid % TPR;
  const floatx4* squares = (const floatx4*)(p.nm.norm_partial + (size_t)min(sq_row, p.M - 1) * p.nm.norm_parts);
  const int fours = p.nm.norm_parts >> 2;
  if (p.nm.norm_partial) {
#pragma unroll
    for (int j = 0; j < 2; ++j) first[j] = squares[min(sq_at + j * TPR, fours - 1)];
  }
  // What the epilogue adds into, gains and bias, as they lie in memory, from rows and columns that are there (a branch of lanes
  // or a conversion would wait for each load): the sums before the first block where this workgroup writes them, else, with the
  // rest, while it counts its arrival. A step of 64 rows (8B) 5,395 -> 5,347 us against requests where they are used, a prompt of 487 rows
  // (0.6B) 2,394 -> 2,361.
  constexpr int IPT = (OT * MT + NW - 1) / NW, MATS = GATED ? 2 : 1;  // a thread's items of four columns of a row
  const bool vec = (p.ldo & 3) == 0 && ((uintptr_t)p.out & 15) == 0;
  floatx4 prev[IPT];
  uint32_t raw_b[IPT][4], raw_eg[IPT][4];
#pragma unroll
  for (int it = 0; it < IPT; ++it) prev[it] = floatx4{0.f, 0.f, 0.f, 0.f};
  auto request_sums = [&]() {
    if (p.epilogue != 1) return;
#pragma unroll
    for (int it = 0; it < IPT; ++it) {
      const int idx = min(tid + it * NW * 64, OT * MT * 64 - 1);
      const float* o = (const float*)p.out + (size_t)min(((idx >> 6) % MT) * 16 + col, p.M - 1) * p.ldo + min(n0 + (idx >> 6) / MT * 16 + g * 4, p.N - 4);
      if (vec)
        prev[it] = *(const floatx4*)o;
      else
        prev[it] = floatx4{o[0], o[1], o[2], o[3]};
    }
  };
  auto request_vector = [&](const void* vector, int dtype, uint32_t (&raw)[IPT][4]) {
    auto entries = [&](auto* v) {
#pragma unroll
      for (int it = 0; it < IPT; ++it) {
        const int n = min(n0 + (min(tid + it * NW * 64, OT * MT * 64 - 1) >> 6) / MT * 16 + g * 4, p.N - 4);
#pragma unroll
        for (int i = 0; i < 4; ++i) raw[it][i] = v[n + i];
      }
    };
    if (dtype == JLLM_BF16)
      entries((const uint16_t*)vector);
    else
      entries((const uint32_t*)vector);
  };
  auto request_vectors = [&]() {
    if (p.nm.emit_rows) request_vector(p.nm.emit_gain, p.nm.emit_gain_dtype, raw_eg);
    if (p.bias) request_vector(p.bias, p.bias_dtype, raw_b);
  };
  constexpr bool AHEAD = GATED || CT < 8 || !SHARED;  // two workgroups of 16 waves: 64 registers a thread, too few for it
  if (AHEAD && parts == 1) request_sums();
  // ---- the loads of a block: 8 weight rows per wave, and 8 activation rows for as many waves as that takes
  const int lrow = lane >> 3, lslot = lane & 7;
  const int na = (p.M + 7) >> 3;
  const int nl = 1 + (na > wave ? (na - wave + NW - 1) / NW : 0);  // the wave's loads per block
  const int wr = wave * 8 + lrow;                                  // row of the block's weights in LDS
  const bool up = GATED && wave >= CT;
  const int wn = min(n0 + (up ? wr - CT * 8 : wr), p.N - 1);
  const uint32_t wlds = (uint32_t)wave * 1024u;
  const uint32_t woff = (uint32_t)(wn - min(n0, p.N - 1)) * (uint32_t)p.K * 2u + (uint32_t)((lslot ^ ring_swz(wr)) * 16);
  const unsigned char* wbase = (const unsigned char*)((up ? p.W2 : p.W) + (size_t)min(n0, p.N - 1) * p.K) + (size_t)b_first * GS_ROW_BYTES;
  const unsigned char* abase = (const unsigned char*)p.A + (size_t)b_first * GS_ROW_BYTES;
  uint32_t aoff[AL];
#pragma unroll
  for (int c = 0; c < AL; ++c) {
    const int r = (wave + c * NW) * 8 + lrow;
    aoff[c] = (uint32_t)min(r, p.M - 1) * (uint32_t)p.lda * 2u + (uint32_t)((lslot ^ ring_swz(r)) * 16);
  }
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)smem;
  auto issue = [&](int i, int slot) {
    const uint32_t at = lds0 + (uint32_t)slot * BLOCK;
    int b = i + rot;
    if (b >= total) b -= total;
    const size_t kbytes = (size_t)b * GS_ROW_BYTES;
    load_to_lds_16(wbase + kbytes, woff, at + wlds);
#pragma unroll
    for (int c = 0; c < AL; ++c)
      if (wave + c * NW < na) load_to_lds_16(abase + kbytes, aoff[c], at + (uint32_t)(2 * CT + wave + c * NW) * 1024u);
  };
#pragma unroll
  for (int i = 0; i < S - 1; ++i)
    if (i < total) issue(i, i);
  // ---- fragments: lane l reads row l % 16, 8 of k at kg * 32 + (l / 16) * 8: piece 4 kg + l / 16
  const int foff = col * GS_ROW_BYTES + (((4 * kg + g) ^ ring_swz(col)) << 4);  // + 16 rows leave ring_swz unchanged
  floatx4 acc[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) acc[m] = floatx4{0.f, 0.f, 0.f, 0.f};
  int slot = 0, fill = S - 1, i = 0;
  auto block = [&]() {  // block i has come to this wave
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the reads of block i - 1, whose slot is filled next
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    if (i + S - 1 < total) issue(i + S - 1, fill);
    const unsigned char* blk = smem + slot * BLOCK + foff;
    const u32x4 w = *(const u32x4*)(blk + ct * 2048);
    u32x4 a[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) a[m] = *(const u32x4*)(blk + (CT + m) * 2048);
    // the weights as the first operand: a lane then holds four consecutive columns of one row
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[m] = mfma16(w, a[m], acc[m]);
    fill = slot;
    if (++slot == S) slot = 0;
  };
  // block i: issued, with S - 2 behind it where there are as many; the wave's own loads, then everybody's. A loop of its own for
  // every number of loads a wave may have (a last tile of few rows leaves some waves without any for it): chosen inside the
  // loop they made products with such a tile slower than full ones (6,144 x 4,096 at 400 rows 49.2 us, at 512 45.0; now 42.3)
  gs_with_loads<1 + AL>(nl, [&](auto loads) {
    for (; i + S - 2 < total; ++i) {
      wait_loads<decltype(loads)::n * (S - 2)>();
      block();
    }
  });
  for (; i < total; ++i) {
    gs_wait_at_most((total - 1 - i) * nl);
    block();
  }
  if (AHEAD && parts == 1) request_vectors();
  if (p.nm.norm_partial) {
    float t = sq_at < fours ? (first[0][0] + first[0][1]) + (first[0][2] + first[0][3]) : 0.f;
    t += sq_at + TPR < fours ? (first[1][0] + first[1][1]) + (first[1][2] + first[1][3]) : 0.f;
    for (int q = sq_at + 2 * TPR; q < (sq_row < p.M ? fours : 0); q += TPR) {
      const floatx4 v = squares[q];
      t += (v[0] + v[1]) + (v[2] + v[3]);
    }
#pragma unroll
    for (int o = 1; o < TPR; o <<= 1) t += __shfl_xor(t, o, 64);
    if (sq_at == 0 && sq_row < p.M) rs[sq_row] = 1.0f / sqrtf(t / (float)p.K + p.nm.norm_eps);
  }
  __syncthreads();  // every wave is done with the ring, which now holds the waves' sums
  floatx4(*red)[CT][MT][64] = (floatx4(*)[CT][MT][64])smem;
#pragma unroll
  for (int m = 0; m < MT; ++m) red[kg][ct][m][lane] = acc[m];
  __syncthreads();
  constexpr int ITEMS = CT * MT * 64;       // a tile's 16 rows by 16 columns are 64 items of four columns
  float* mine = p.partial + tile * parts * ITEMS * 4;
  if (parts > 1) {
    for (int idx = tid; idx < ITEMS; idx += NW * 64) {
      if (((idx >> 6) % MT) * 16 + (idx & 15) >= p.M) continue;
      const floatx4 v = (&red[0][0][0][0])[idx] + (&red[1][0][0][0])[idx];
      float* dst = mine + ((size_t)blockIdx.y * ITEMS + idx) * 4;
      store_shared2(dst, v[0], v[1]);
      store_shared2(dst + 2, v[2], v[3]);
    }
    shared_stores_done();
    if (AHEAD) {
      request_sums();
      request_vectors();
    }
    __syncthreads();
    if (tid == 0) last = arrived_last(p.arrivals + tile, parts);
    __syncthreads();
    if (!last) return;
  }
  // a thread's items (64 lanes of a wave: one tile, one tile of rows): everything they read is requested side by side
  floatx4 sum[IPT][MATS];
#pragma unroll
  for (int it = 0; it < IPT; ++it)
#pragma unroll
    for (int u = 0; u < MATS; ++u) sum[it][u] = floatx4{0.f, 0.f, 0.f, 0.f};
  if (parts == 1) {
#pragma unroll
    for (int it = 0; it < IPT; ++it)
#pragma unroll
      for (int u = 0; u < MATS; ++u) {
        const int idx = min(tid + it * NW * 64, OT * MT * 64 - 1) + u * OT * MT * 64;
        sum[it][u] = (&red[0][0][0][0])[idx] + (&red[1][0][0][0])[idx];
      }
  } else {
    constexpr int Z = IPT * MATS > 2 ? 2 : 4;  // so many parts of every item are requested before any is added
    for (int z0 = 0; z0 < parts; z0 += Z) {
      floatx4 q[Z][IPT][MATS];
#pragma unroll
      for (int z = 0; z < Z; ++z)
#pragma unroll
        for (int it = 0; it < IPT; ++it)
#pragma unroll
          for (int u = 0; u < MATS; ++u) {
            int idx = min(tid + it * NW * 64, OT * MT * 64 - 1) + u * OT * MT * 64;
            if (((idx >> 6) % MT) * 16 + col >= p.M) idx = 0;  // a row that is not there: any that is
            const float* src = mine + ((size_t)min(z0 + z, parts - 1) * ITEMS + idx) * 4;
            float x0, x1, x2, x3;
            load_shared2(src, x0, x1);
            load_shared2(src + 2, x2, x3);
            q[z][it][u] = floatx4{x0, x1, x2, x3};
          }
#pragma unroll
      for (int z = 0; z < Z; ++z)
        if (z0 + z < parts) {
#pragma unroll
          for (int it = 0; it < IPT; ++it)
#pragma unroll
            for (int u = 0; u < MATS; ++u) sum[it][u] += q[z][it][u];
        }
    }
  }
  if (!AHEAD) {
    request_sums();
    request_vectors();
  }
#pragma unroll
  for (int it = 0; it < IPT; ++it) {
    const int idx = tid + it * NW * 64;
    if (idx >= OT * MT * 64) continue;
    const int t = (idx >> 6) / MT, m = ((idx >> 6) % MT) * 16 + col;
    const int n = n0 + t * 16 + g * 4;
    float sq = 0.f;
    if (m < p.M && n < p.N) {
      const size_t o = (size_t)m * p.ldo + n;
      const float scale = p.nm.norm_partial ? rs[m] : 1.0f;
      float r[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float x = sum[it][0][i] * scale;
        if (p.bias) x += raw_value(raw_b[it][i], p.bias_dtype);
        if (GATED) x = gated<false>(x, sum[it][MATS - 1][i] * scale, p.gate);
        r[i] = prev[it][i] + x;
        sq += r[i] * r[i];
      }
      if (p.nm.emit_rows) {
        float e[4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
          e[i] = r[i] * raw_value(raw_eg[it][i], p.nm.emit_gain_dtype);
        *(u32x2*)(p.nm.emit_rows + (size_t)m * p.nm.emit_ld + n) = u32x2{pack_bf16(e[0], e[1]), pack_bf16(e[2], e[3])};
      }
      if (p.out_dtype == JLLM_BF16) {
        if (vec)
          *(u32x2*)((bf16_t*)p.out + o) = u32x2{pack_bf16(r[0], r[1]), pack_bf16(r[2], r[3])};
        else
#pragma unroll
          for (int i = 0; i < 4; ++i) stf((bf16_t*)p.out, o + i, r[i]);
      } else {
        if (vec)
          *(floatx4*)((float*)p.out + o) = floatx4{r[0], r[1], r[2], r[3]};
        else
#pragma unroll
          for (int i = 0; i < 4; ++i) ((float*)p.out)[o + i] = r[i];
      }
    }
    if (p.nm.emit_rows) {  // over the lanes of one row
      sq += __shfl_xor(sq, 16, 64);
      sq += __shfl_xor(sq, 32, 64);
      if (g == 0) rowsq[t][m] = sq;
    }
  }
  if (p.nm.emit_rows) {
    __syncthreads();
    const int spare = p.nm.emit_parts - (int)gridDim.x;
    for (int m = tid; m < p.M; m += NW * 64) {
      float t = 0.f;
#pragma unroll
      for (int c = 0; c < OT; ++c) t += rowsq[c][m];
      float* dst = p.nm.emit_partial + (size_t)m * p.nm.emit_parts;
      dst[blockIdx.x] = t;
      for (int z = blockIdx.x; z < spare; z += gridDim.x) dst[gridDim.x + z] = 0.f;
    }
  }
}

template <int CT, int MT, bool GATED, bool SHARED>
static int launch_stream(const StreamArgs& a, dim3 grid, hipStream_t stream) {
  constexpr size_t smem = (size_t)gs_slots(CT, MT, SHARED) * (2 * CT + 2 * MT) * 1024;
  static bool configured = false;
  if (!configured) {  // above 64 KB the size has to be allowed first
    if (hipFuncSetAttribute((const void*)gemm_stream_kernel<CT, MT, GATED, SHARED>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem) != hipSuccess)
      JLLM_FAIL("gemm_stream: cannot reserve %zu bytes of LDS", smem);
    configured = true;
  }
  gemm_stream_kernel<CT, MT, GATED, SHARED><<<grid, CT * 128, smem, stream>>>(a);
  JLLM_CHECK_LAUNCH("gemm_stream");
  return 0;
}

template <int CT, bool GATED>
static int launch_stream_rows(const StreamArgs& a, dim3 grid, int row_tiles, bool shared, hipStream_t stream) {
#define GS_CASE(MT)                                                       \
  case MT:                                                                \
    return shared ? launch_stream<CT, MT, GATED, true>(a, grid, stream) : launch_stream<CT, MT, GATED, false>(a, grid, stream);
  switch (row_tiles) {
    GS_CASE(2) GS_CASE(3) GS_CASE(4)
    default: return launch_stream<CT, 8, GATED, false>(a, grid, stream);
  }
#undef GS_CASE
}

// `rows`: weight rows per workgroup, both weights' of the gated epilogue together (32, 64, 96 or 128). `tile_m`: activation
// rows per workgroup (64 or 128; up to 64 rows in all take tiles of 32, 48 or 64). `parts` > 1 cuts K over
// gridDim.y in whole blocks of 128; `partial` then holds parts * column tiles * rows * (tiles of rows in all) * (their rows) floats and `arrivals`
// one int per column tile (and tile of rows), zeros, left as zeros. An RMSNorm on either side as in jllm_gemm_skinny_norm_bf16.
// returns 0 when it ran, 1 when the shape is not one it takes (the caller uses another kernel), -1 on errors
extern "C" int jllm_gemm_stream_bf16(const void* A, int lda, const void* W, const void* W2, const void* bias,
                                     int bias_dtype, void* out, int out_dtype, int ldo, int M, int N, int K, int epilogue,
                                     float gate_limit, int rows, int tile_m, int parts, float* partial, int* arrivals, void* emit_rows, int emit_ld,
                                     const void* emit_gain, int emit_gain_dtype, float* emit_partial, int emit_parts,
                                     const float* norm_partial, int norm_parts, float norm_eps, hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if ((K & 127) || (N & 15) || (lda & 7) || K <= 0 || lda < 0) return 1;
  if (((uintptr_t)A & 15) || ((uintptr_t)W & 15) || (W2 && ((uintptr_t)W2 & 15))) return 1;
  if (tile_m != 64 && tile_m != 128) JLLM_FAIL("gemm_stream: tiles of %d rows (64 and 128)", tile_m);
  // a lane's place in an operand is a 32-bit byte offset from the workgroup's first row
  if ((unsigned long long)lda >= (1ull << 24) || (unsigned long long)K >= (1ull << 23)) return 1;
  JLLM_TAKE_GATE("gemm_stream", epilogue, gate_limit, gs);
  if (epilogue < 0 || epilogue > 2 || (epilogue == 2) != (W2 != nullptr)) JLLM_FAIL("gemm_stream: epilogue %d", epilogue);
  if (epilogue == 1 && out_dtype != JLLM_F32) JLLM_FAIL("gemm_stream: the accumulate epilogue adds into fp32");
  if (ldo < N) JLLM_FAIL("gemm_stream: ldo %d < N %d", ldo, N);
  if (rows != 32 && rows != 64 && rows != 96 && rows != 128) JLLM_FAIL("gemm_stream: %d weight rows per workgroup (32, 64, 96, 128)", rows);
  const int cols = W2 ? rows / 2 : rows;
  const int tiles = (N + cols - 1) / cols;
  const int nblk = K >> 7;
  if (parts < 1) parts = 1;
  if (parts > nblk) parts = nblk;
  const int bpp = (nblk + parts - 1) / parts;
  const int used = (nblk + bpp - 1) / bpp;  // parts that have any block
  if (used > 1 && (!partial || !arrivals || ((uintptr_t)partial & 15))) JLLM_FAIL("gemm_stream: %d parts of K need a buffer for their sums and counters", used);
  if (emit_rows && (epilogue != 1 || !emit_gain || !emit_partial)) JLLM_FAIL("gemm_stream: rows for a norm come from the accumulate epilogue, with gain and partial sums");
  if (emit_rows && (emit_ld < N || (emit_ld & 3) || ((uintptr_t)emit_rows & 7))) JLLM_FAIL("gemm_stream: rows for a norm with stride %d", emit_ld);
  if (emit_rows && emit_parts < tiles) JLLM_FAIL("gemm_stream: %d places for the partial sums of %d workgroups", emit_parts, tiles);
  if (norm_partial && norm_parts <= 0) JLLM_FAIL("gemm_stream: %d partial sums", norm_parts);
  if (norm_partial && ((norm_parts & 3) || ((uintptr_t)norm_partial & 15))) return 1;
  const int cus = jllm_compute_units();
  if (cus <= 0) JLLM_FAIL("gemm_stream: the GPU's compute units could not be read");
  dim3 grid(tiles, used, (M + tile_m - 1) / tile_m);
  if (grid.y > 65535 || grid.z > 65535) return 1;
  const int row_tiles = M > 64 ? tile_m / 16 : M > 32 ? (M + 15) / 16 : 2;
  const StreamArgs a{(const bf16_t*)A, (const bf16_t*)W, (const bf16_t*)W2, bias, out, partial, arrivals, lda, bias_dtype, out_dtype, ldo, M, N, K,
                     epilogue, bpp * 2, M <= 64 && used == 1, gs, StreamNorm{(bf16_t*)emit_rows, emit_ld, emit_gain, emit_gain_dtype, emit_partial, emit_parts, norm_partial, norm_parts, norm_eps}};
  // two workgroups share a compute unit where there are more of them than compute units: one streams while the other adds up
  const bool shared = (long)tiles * used * grid.z > cus;
  if (W2) switch (rows) {
      case 32: return launch_stream_rows<2, true>(a, grid, row_tiles, shared, stream);
      case 64: return launch_stream_rows<4, true>(a, grid, row_tiles, shared, stream);
      case 96: return launch_stream_rows<6, true>(a, grid, row_tiles, shared, stream);
      default: return launch_stream_rows<8, true>(a, grid, row_tiles, shared, stream);
    }
  switch (rows) {
    case 32: return launch_stream_rows<2, false>(a, grid, row_tiles, shared, stream);
    case 64: return launch_stream_rows<4, false>(a, grid, row_tiles, shared, stream);
    case 96: return launch_stream_rows<6, false>(a, grid, row_tiles, shared, stream);
    default: return launch_stream_rows<8, false>(a, grid, row_tiles, shared, stream);
  }
}
