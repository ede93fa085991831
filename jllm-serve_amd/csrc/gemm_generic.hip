// C[M,N] = A[M,K] * W[N,K]^T for any sizes and for fp32 or bf16 operands (widened), every sum in true fp32: the 32-bit path
// of every linear layer, and the fallback for shapes the bf16 matrix-core kernels refuse.
//
// The products run on the matrix cores' fp32 form, v_mfma_f32_16x16x4_f32, which rounds after every multiply-add and
// takes its four k in ascending order: an output is the same bits as one accumulator walked with fmaf from k = 0 to
// K - 1 (compared bit for bit on the GPU, also for sums that end in denormals). So an output never depends on M, on the
// other rows of the batch or on which of the two kernels below computed it, and K is never cut. The vector units, which
// this project builds without their packed fp32 forms, reach half the matrix cores' fp32 rate.
//
// Fragments: lane l of the MFMA holds row l % 16 at k = 4 s + l / 16 of step s. Memory holds a row's k side by side, so 16
// bytes of a lane (k = 4 q .. 4 q + 3, q = l / 16) are one step's values of four lane groups, and a lane wants one value of
// four steps: a transposition of 4 x 4 over the lane groups, done as the operands are written to LDS.
//
// Epilogues: 0 store (fp32 or bf16), 1 add into an fp32 matrix (the residual stream), 2 gated:
// out = gate(A*Wg^T, A*Wu^T) (the gate functions of common.h) with two weight matrices sharing the A tile.
#include "common.h"
#include "layer_launches.h"
#include "lds_ring.h"

typedef float floatx4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ floatx4 mfma_f32(float w, float a, floatx4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(w, a, c, 0, 0, 0);
}

// bias, gate and store of one output
template <bool GATED>
__device__ __forceinline__ void finish_output(float v, float up, int m, int n, const void* __restrict__ bias, int bias_dtype,
                                              void* __restrict__ out, int out_dtype, int ldo, int epilogue, GateSpec gs) {
  if (bias) v += (bias_dtype == JLLM_BF16) ? ldf((const bf16_t*)bias, n) : ldf((const float*)bias, n);
  const size_t o = (size_t)m * ldo + n;
  if (GATED) {
    const float g = v;
    v = gated<false>(g, up, gs);
  }
  if (epilogue == 1) {
    ((float*)out)[o] += v;
  } else if (out_dtype == JLLM_BF16) {
    stf((bf16_t*)out, o, v);
  } else {
    stf((float*)out, o, v);
  }
}

// four neighbouring outputs of one row: as finish_output, with one access where all four exist and lie on a boundary
template <bool GATED>
__device__ __forceinline__ void finish_four(floatx4 v, floatx4 u, int m, int n, int N, const void* __restrict__ bias, int bias_dtype,
                                            void* __restrict__ out, int out_dtype, int ldo, int epilogue, GateSpec gs) {
  if (n + 3 < N && out_dtype == JLLM_F32 && (ldo & 3) == 0 && (((uintptr_t)out) & 15) == 0) {
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      if (bias) v[c] += (bias_dtype == JLLM_BF16) ? ldf((const bf16_t*)bias, n + c) : ldf((const float*)bias, n + c);
      if (GATED) v[c] = gated<false>(v[c], u[c], gs);
    }
    floatx4* o = (floatx4*)((float*)out + (size_t)m * ldo + n);
    if (epilogue == 1) {
      const floatx4 cur = *o;
#pragma unroll
      for (int c = 0; c < 4; ++c) v[c] = cur[c] + v[c];
    }
    *o = v;
    return;
  }
#pragma unroll
  for (int c = 0; c < 4; ++c)
    if (n + c < N) finish_output<GATED>(v[c], u[c], m, n + c, bias, bias_dtype, out, out_dtype, ldo, epilogue, gs);
}

// four consecutive elements of a row as floats. WIDE: k and K are multiples of four and the row starts on a boundary of
// four elements; else element by element. Beyond K: zeros, which add nothing to a sum (in both operands, so that an
// infinity in the other one is not multiplied by them).
__device__ __forceinline__ floatx4 widen(floatx4 v) { return v; }
__device__ __forceinline__ floatx4 widen(uint2 t) {
  return floatx4{__uint_as_float(t.x << 16), __uint_as_float(t.x & 0xffff0000u), __uint_as_float(t.y << 16), __uint_as_float(t.y & 0xffff0000u)};
}
template <typename T>
struct Four;  // four elements as they lie in memory
template <>
struct Four<float> {
  typedef floatx4 type;
};
template <>
struct Four<bf16_t> {
  typedef uint2 type;
};
template <typename T, bool WIDE>
__device__ __forceinline__ floatx4 load4k(const T* __restrict__ row, int k, int K) {
  if (WIDE) {
    const floatx4 v = widen(*(const typename Four<T>::type*)(row + (k < K ? k : 0)));
    return k < K ? v : floatx4{0.f, 0.f, 0.f, 0.f};
  }
  floatx4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int j = 0; j < 4; ++j)
    if (k + j < K) v[j] = ldf(row, k + j);
  return v;
}
// a piece of a stage in registers: four elements as they lie in memory, or, where rows cannot be read four at a time, as floats
template <typename T, bool WIDE>
struct Piece {
  typedef typename Four<T>::type type;
  static __device__ __forceinline__ type load(const T* __restrict__ row, int k, int K) { return *(const type*)(row + (k < K ? k : 0)); }
  static __device__ __forceinline__ floatx4 value(type v, bool in) { return in ? widen(v) : floatx4{0.f, 0.f, 0.f, 0.f}; }
};
template <typename T>
struct Piece<T, false> {
  typedef floatx4 type;
  static __device__ __forceinline__ type load(const T* __restrict__ row, int k, int K) { return load4k<T, false>(row, k, K); }
  static __device__ __forceinline__ floatx4 value(type v, bool) { return v; }
};

// Many rows: a workgroup of WM x WN waves owns a tile of 16 WM FM rows by 16 WN FN outputs, a wave FM x FN accumulators of
// 16 x 16. Eight waves (two on every SIMD) where the tile has work for them: a wave alone on its SIMD multiplies nothing
// while it reads and writes LDS.
// K advances in stages of BK through two LDS buffers, the operands of the next two stages on their way into registers while
// one is multiplied. LDS holds blocks of 16 rows x 16 k in the order the lanes read them (lane l's 16 bytes: its row at
// k = q, 4 + q, 8 + q, 12 + q), so a fragment read is 1 KB side by side and the four 4-byte writes of a thread's 16
// bytes go to neighbouring words across the wave.
template <typename TA, typename TW, bool GATED, int WM, int WN, int FM, int FN, int BK, bool WIDE>
__global__ __launch_bounds__(WM * WN * 64) void gemm_f32_tile_kernel(const TA* __restrict__ A, int lda, const TW* __restrict__ W,
                                                            const TW* __restrict__ W2, const void* __restrict__ bias,
                                                            int bias_dtype, void* __restrict__ out, int out_dtype, int ldo,
                                                            int M, int N, int K, int epilogue, GateSpec gs) {
  constexpr int TM = WM * FM * 16, TN = WN * FN * 16, NW = GATED ? 2 : 1, TH = WM * WN * 64;
  constexpr int ROWS = TM + NW * TN, CH = BK / 16, QPR = BK / 4;  // rows staged, 16-k chunks and 16-byte pieces per row
  constexpr int UA = TM * QPR / TH, UW = NW * TN * QPR / TH;      // pieces per thread and stage
  static_assert(TM * QPR % TH == 0 && TN * QPR % TH == 0, "whole pieces of one operand per thread");
  extern __shared__ __align__(16) float lds[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WN, wn = wave % WN;
  const int m0 = blockIdx.y * TM, n0 = blockIdx.x * TN;
  // a stage's pieces on their way: as memory holds them (widened, and zeroed beyond K, when they are written to LDS), so
  // that nothing waits for a load before its stage
  struct Set {
    typename Piece<TA, WIDE>::type a[UA];
    typename Piece<TW, WIDE>::type w[UW];
  };
  const int pr = tid / QPR, pk = (tid % QPR) * 4;  // this thread's row (+ TH / QPR per piece) and place in a stage's k
  auto fetch = [&](Set& st, int k0) {
#pragma unroll
    for (int i = 0; i < UA; ++i)
      st.a[i] = Piece<TA, WIDE>::load(A + (size_t)min(m0 + pr + i * (TH / QPR), M - 1) * lda, k0 + pk, K);
#pragma unroll
    for (int i = 0; i < UW; ++i) {  // which weight a piece belongs to is the same for all threads
      const int r = pr + (i % (UW / NW)) * (TH / QPR);
      st.w[i] = Piece<TW, WIDE>::load((i < UW / NW ? W : W2) + (size_t)min(n0 + r, N - 1) * K, k0 + pk, K);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  auto put = [&](const Set& st, int buf, int k0) {
    const bool in = k0 + pk < K;
    float* base = lds + buf * ROWS * BK + (pk >> 4) * 256;
    const int turn = (pk >> 4) * (64 / CH);
#pragma unroll
    for (int i = 0; i < UA + UW; ++i) {
      const floatx4 v = i < UA ? Piece<TA, WIDE>::value(st.a[i < UA ? i : 0], in) : Piece<TW, WIDE>::value(st.w[i < UA ? 0 : i - UA], in);
      const int r = pr + i * (TH / QPR);
      float* dst = base + (r >> 4) * CH * 256 + (((r & 15) * 4 + ((pk >> 2) & 3)) ^ turn);
#pragma unroll
      for (int j = 0; j < 4; ++j) dst[j * 64] = v[j];
    }
  };
  floatx4 acc[NW][FM][FN];
#pragma unroll
  for (int w = 0; w < NW; ++w)
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j) acc[w][i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
  auto multiply = [&](int buf) {
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      const float* at = lds + buf * ROWS * BK + ((lane * 4) ^ (c * (64 / CH)));
      floatx4 a[FM], w[NW][FN];
#pragma unroll
      for (int i = 0; i < FM; ++i) a[i] = *(const floatx4*)(at + ((wm * FM + i) * CH + c) * 256);
#pragma unroll
      for (int z = 0; z < NW; ++z)
#pragma unroll
        for (int j = 0; j < FN; ++j) w[z][j] = *(const floatx4*)(at + ((WM * FM + (z * WN + wn) * FN + j) * CH + c) * 256);
#pragma unroll
      for (int q = 0; q < 4; ++q)  // k = 16 c + 4 q .. + 3
#pragma unroll
        for (int z = 0; z < NW; ++z)
#pragma unroll
          for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j) acc[z][i][j] = mfma_f32(w[z][j][q], a[i][q], acc[z][i][j]);
    }
  };
  const int stages = (K + BK - 1) / BK;
  Set s0, s1;
  fetch(s0, 0);
  fetch(s1, BK);
  put(s0, 0, 0);
  __syncthreads();
  for (int s = 0; s < stages; s += 2) {
    fetch(s0, (s + 2) * BK);  // beyond the end: some place inside the rows, never multiplied
    multiply(0);
    put(s1, 1, (s + 1) * BK);
    __syncthreads();
    if (s + 1 >= stages) break;
    fetch(s1, (s + 3) * BK);
    multiply(1);
    put(s0, 0, (s + 2) * BK);
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < FM; ++i) {
    const int m = m0 + (wm * FM + i) * 16 + (lane & 15);
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      const int n = n0 + (wn * FN + j) * 16 + (lane >> 4) * 4;
      if (m < M) finish_four<GATED>(acc[0][i][j], acc[NW - 1][i][j], m, n, N, bias, bias_dtype, out, out_dtype, ldo, epilogue, gs);
    }
  }
}

// The same tiles with fp32 operands whose rows are whole lines (K a multiple of 32, rows on 16 bytes): stages of 32 k go straight from
// memory into a ring of RING places in LDS (lds_ring.h), RING - 1 of them on their way. Nothing is transposed on the way: a step of a
// fragment is one word a lane, and of the rows of 128 bytes with their pieces turned by ring_swz the 64 words that a read names (16
// rows at k = 4 s .. 4 s + 3) fall into all 64 banks. One barrier a stage, two steps before the stage ends: in front of it a wave waits
// for its own share of the next stage, behind it the place of the stage before is asked for again, and the next stage's first fragments
// are read while the last steps are multiplied. The sums are those of the kernel above, bit for bit.
// It is bound by the matrix cores (32 cycles a step and accumulator: 157 TFLOP/s) and by what rounds of workgroups leave idle; the kernel
// above also waits for its four 4-byte writes to LDS for every 16 bytes, and once a step for its fragments. us, the kernel above / this:
// 1,000 rows of 4,096 x 1,024 76.6 / 65.9, of 4,096 x 2,048 146 / 125 (134 TFLOP/s), of 1,024 x 3,072 68.6 / 52.4, gated 3,072 x 1,024
// 119.7 / 101.3; 487 of 2,048 x 6,144 132 / 101, of 1,024 x 2,048 (32 x 32) 29.6 / 22.9; 40 rows of 1,024 x 3,072 28.1 / 25.1 (a chain of
// 768 steps, three times its cycles: four waves alone on a compute unit, bound by the wait for memory). With the barrier behind the last step and the
// compiler's own order of reads and multiplies: 71.6, 137, 65.3, 113.9.
template <bool GATED, int WM, int WN, int FM, int FN, int RING>
__global__ __launch_bounds__(WM * WN * 64) void gemm_f32_ring_kernel(const float* __restrict__ A, int lda, const float* __restrict__ W,
                                                            const float* __restrict__ W2, const void* __restrict__ bias,
                                                            int bias_dtype, void* __restrict__ out, int out_dtype, int ldo,
                                                            int M, int N, int K, int epilogue, GateSpec gs) {
  constexpr int TM = WM * FM * 16, TN = WN * FN * 16, NW = GATED ? 2 : 1;
  constexpr int ROWS = TM + NW * TN, STAGE = ROWS * 32;  // rows of a stage; floats of one place of the ring
  constexpr int LOADS = ROWS / 8 / (WM * WN);            // of 1 KB, eight rows each, per wave and stage
  static_assert(ROWS % (8 * WM * WN) == 0 && RING >= 3 && RING <= 8, "whole loads per wave");
  extern __shared__ __align__(1024) float lds[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave / WN, wn = wave % WN;
  const int m0 = blockIdx.y * TM, n0 = blockIdx.x * TN;
  const int stages = K / 32;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) float*)lds;
  const float* at[LOADS];  // this lane's piece of each of the wave's loads of the next stage
#pragma unroll
  for (int i = 0; i < LOADS; ++i) {
    const int row = (wave * LOADS + i) * 8 + (lane >> 3);  // the tile's rows: A, then W, then W2
    const int piece = (lane & 7) ^ ring_swz(row & 15);
    const int r = row - TM, n = min(n0 + (r >= TN ? r - TN : r), N - 1);
    at[i] = (row < TM ? A + (size_t)min(m0 + row, M - 1) * lda : (GATED && r >= TN ? W2 : W) + (size_t)n * K) + piece * 4;
  }
  auto issue = [&](int place) {
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      load_to_lds_16(at[i], lds0 + (uint32_t)(place * STAGE * 4 + (wave * LOADS + i) * 1024));
      at[i] += 32;
    }
  };
  floatx4 acc[NW][FM][FN];
#pragma unroll
  for (int z = 0; z < NW; ++z)
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j) acc[z][i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
  const int fr = lane & 15;
  const float* word[8];  // of step s: row `fr`, k = 4 s + lane / 16 of the first block of a place
#pragma unroll
  for (int s = 0; s < 8; ++s) word[s] = lds + fr * 32 + ((s ^ ring_swz(fr)) << 2) + (lane >> 4);
  // A step's fragments are asked for two steps ahead, also across stages (behind the last one what lies in the ring, which nothing
  // multiplies), and the compiler is held to that order: left to itself it reads in front of the use and waits there.
  float a[4][FM], w[4][NW][FN];
  auto read = [&](int place, int s) {
#pragma unroll
    for (int i = 0; i < FM; ++i) a[s & 3][i] = word[s][place * STAGE + (wm * FM + i) * 512];
#pragma unroll
    for (int z = 0; z < NW; ++z)
#pragma unroll
      for (int j = 0; j < FN; ++j) w[s & 3][z][j] = word[s][place * STAGE + TM * 32 + ((z * WN + wn) * FN + j) * 512];
  };
  auto landed = [&](int behind) {  // what is next is there for all waves, with so many stages behind it still on their way
    switch (min(RING - 2, behind)) {
      case 6: wait_loads<6 * LOADS>(); break;
      case 5: wait_loads<5 * LOADS>(); break;
      case 4: wait_loads<4 * LOADS>(); break;
      case 3: wait_loads<3 * LOADS>(); break;
      case 2: wait_loads<2 * LOADS>(); break;
      case 1: wait_loads<1 * LOADS>(); break;
      default: wait_loads<0>();
    }
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
#pragma unroll
  for (int t = 0; t < RING - 1; ++t)
    if (t < stages) issue(t);
  landed(stages - 1);
  read(0, 0);
  read(0, 1);
  for (int t0 = 0; t0 < stages; t0 += RING) {
#pragma unroll
    for (int place = 0; place < RING; ++place) {
      const int t = t0 + place;
      if (t >= stages) break;
#pragma unroll
      for (int s = 0; s < 8; ++s) {  // k = 32 t + 4 s .. + 3
        if (s == 6 && t + 1 < stages) {
          landed(min(RING - 3, stages - 2 - t));
          if (t + RING - 1 < stages) issue((place + RING - 1) % RING);  // where stage t - 1 was: all waves are in stage t
        }
        read(s < 6 ? place : (place + 1) % RING, (s + 2) & 7);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int z = 0; z < NW; ++z)
#pragma unroll
          for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j) acc[z][i][j] = mfma_f32(w[s & 3][z][j], a[s & 3][i], acc[z][i][j]);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }
#pragma unroll
  for (int i = 0; i < FM; ++i) {
    const int m = m0 + (wm * FM + i) * 16 + fr;
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      const int n = n0 + (wn * FN + j) * 16 + (lane >> 4) * 4;
      if (m < M) finish_four<GATED>(acc[0][i][j], acc[NW - 1][i][j], m, n, N, bias, bias_dtype, out, out_dtype, ldo, epilogue, gs);
    }
  }
}

// Up to 16 rows (decode steps of the 32-bit path). An output's chain is 8 cycles per k (a 16 x 16 x 4 product takes 32), so
// a product of few weight rows is bound by that chain (3,072 k: 11 us) as long as nothing else stands in it: a workgroup
// owns 16 weight rows and all activation rows, one wave (two with the gated epilogue, one per weight matrix) does nothing
// but read fragments from LDS and multiply, and three others keep two turns of 16 CH k on their way from memory (1 KB of
// weights per instruction: 16 rows x 64 bytes) and write the turn that arrived to LDS, transposed, in the half that is
// not being multiplied. One wave that loads, transposes with lane swaps (v_permlane16/32_swap) and multiplies took twice
// the chain.
template <typename TA, typename TW, bool GATED, bool WIDE>
__global__ __launch_bounds__(GATED ? 320 : 256) void gemm_f32_rows_kernel(const TA* __restrict__ A, int lda, const TW* __restrict__ W,
                                                                        const TW* __restrict__ W2, const void* __restrict__ bias,
                                                                        int bias_dtype, void* __restrict__ out, int out_dtype,
                                                                        int ldo, int M, int N, int K, int epilogue, GateSpec gs) {
  constexpr int NC = GATED ? 2 : 1, CPP = GATED ? 3 : 4, CH = 3 * CPP;  // multiplying waves; chunks of 16 k per loading wave, per turn
  __shared__ __align__(16) float lds[2][CH][NC + 1][256];             // a chunk's activations, then its weights
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n0 = blockIdx.x * 16;
  const int r = lane & 15, quad = lane >> 4;
  const int turns = (K + CH * 16 - 1) / (CH * 16);
  if (wave >= NC) {
    const int c0 = (wave - NC) * CPP;
    const TA* arow = A + (size_t)min(r, M - 1) * lda;
    const TW* wrow = W + (size_t)min(n0 + r, N - 1) * K;
    const TW* urow = GATED ? W2 + (size_t)min(n0 + r, N - 1) * K : wrow;
    struct Set {
      typename Piece<TA, WIDE>::type a[CPP];
      typename Piece<TW, WIDE>::type w[CPP * NC];
    };
    auto fetch = [&](Set& st, int t) {  // beyond the end: some place inside the rows, never multiplied
#pragma unroll
      for (int c = 0; c < CPP; ++c) {
        const int k = (t * CH + c0 + c) * 16 + quad * 4;
        st.w[c] = Piece<TW, WIDE>::load(wrow, k, K);
        if (GATED) st.w[CPP * (NC - 1) + c] = Piece<TW, WIDE>::load(urow, k, K);
        st.a[c] = Piece<TA, WIDE>::load(arow, k, K);
      }
      __builtin_amdgcn_sched_barrier(0);
    };
    auto put = [&](const Set& st, int t) {
#pragma unroll
      for (int c = 0; c < CPP; ++c) {
        const bool in = (t * CH + c0 + c) * 16 + quad * 4 < K;
#pragma unroll
        for (int z = 0; z <= NC; ++z) {
          const floatx4 v = z == 0 ? Piece<TA, WIDE>::value(st.a[c], in) : Piece<TW, WIDE>::value(st.w[(z ? z - 1 : 0) * CPP + c], in);
          float* dst = &lds[t & 1][c0 + c][z][r * 4 + quad];
#pragma unroll
          for (int j = 0; j < 4; ++j) dst[j * 64] = v[j];  // k = 4 quad + j: step `quad` of lane group j
        }
      }
    };
    Set s0, s1;
    fetch(s0, 0);
    fetch(s1, 1);
    put(s0, 0);
    __syncthreads();
    for (int t = 0; t < turns; t += 2) {
      fetch(s0, t + 2);
      put(s1, t + 1);
      __syncthreads();
      if (t + 1 >= turns) break;
      fetch(s1, t + 3);
      put(s0, t + 2);
      __syncthreads();
    }
    if (GATED) __syncthreads();
    return;
  }
  floatx4 acc = {0.f, 0.f, 0.f, 0.f};
  __syncthreads();
  for (int t = 0; t < turns; ++t) {
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      const floatx4 a = *(const floatx4*)&lds[t & 1][c][0][lane * 4], w = *(const floatx4*)&lds[t & 1][c][1 + wave][lane * 4];
#pragma unroll
      for (int q = 0; q < 4; ++q) acc = mfma_f32(w[q], a[q], acc);
    }
    __syncthreads();
  }
  floatx4 up = acc;
  if (GATED) {
    floatx4* meet = (floatx4*)&lds[0][0][0][0];  // the last turn has been read
    if (wave) meet[lane] = acc;
    __syncthreads();
    if (wave) return;
    up = meet[lane];
  }
  const int n = n0 + quad * 4;
  if (r < M) finish_four<GATED>(acc, up, r, n, N, bias, bias_dtype, out, out_dtype, ldo, epilogue, gs);
}

// Up to four rows, fp32 operands: the same chains on the vector units, where a multiply-add takes 4 cycles and not 8. A lane owns one
// output (16 weight rows x 4 activation rows per wave; gate and up are a wave each), so that nothing but its own chain orders its
// sums. A wave issues one instruction every 4 cycles, so what the chain needs besides has to be little: the four lanes of a
// weight row hold four pieces of it, 16 k in all, from one LDS read, and a multiply-add takes its weight from the quad's lane q by
// DPP; the activations are a read per four k.
// Four other waves keep the operands on their way, straight from memory into a ring of turns of 128 k in LDS. One barrier a turn:
// in front of it the loading waves wait for their part of the turn, behind it they refill the turn that was read before. us inside
// a graph at three rows, the kernel above / this: 4,096 x 2,048 15.1 / 9.9, 1,024 x 2,048 12.7 / 8.8, 1,024 x 3,072 19.0 / 12.3,
// 2,048 x 6,144 35.0 / 22.4 (3.3 ns a k, where the kernel above takes 5.3), gated 3,072 x 1,024 14.4 / 7.9, gated 6,144 x 2,048
// 42.4 / 20.2, 151,936 x 1,024 160 / 107 (5.8 TB/s). Turns of 256 k in a ring of six (144 KB): 7 to 17 % slower, twice as slow
// where compute units then hold one workgroup instead of three.
template <bool GATED>
struct F32Few {
  static constexpr int NC = GATED ? 2 : 1, LOADERS = 4;
  static constexpr int BLOCKS = 4, RING = GATED ? 3 : 4;  // blocks of 32 k per turn, turns
  static constexpr int BLOCK_KB = 2 * NC + 1, TURN_KB = BLOCKS * BLOCK_KB;
  static constexpr int LOADS = TURN_KB / LOADERS;  // of 1 KB: 8 rows x 128 bytes
  static constexpr int THREADS = (NC + LOADERS) * 64;
  static constexpr size_t LDS = (size_t)RING * TURN_KB * 1024;
  static_assert(TURN_KB % LOADERS == 0 && RING * LOADS < 63, "whole loads per wave, as many in flight as the counter holds");
};
// sixteen links of a chain: k = 4 q + j takes w[j] of the quad's lane q and a[q][j]. Written as instructions, which the compiler
// would each make two of (a move by DPP, then the multiply-add); what a DPP operand needs between it and a vector instruction
// that wrote it is waited for here, since the compiler does not look into this.
__device__ __forceinline__ float chain16(floatx4 w, const floatx4 (&a)[4], float acc) {
#define LINK(W, A, Q) "v_fmac_f32_dpp %0, %" #W ", %" #A " quad_perm:[" #Q "," #Q "," #Q "," #Q "] row_mask:0xf bank_mask:0xf\n\t"
  asm("s_nop 1\n\t" LINK(1, 5, 0) LINK(2, 6, 0) LINK(3, 7, 0) LINK(4, 8, 0) LINK(1, 9, 1) LINK(2, 10, 1) LINK(3, 11, 1) LINK(4, 12, 1)
          LINK(1, 13, 2) LINK(2, 14, 2) LINK(3, 15, 2) LINK(4, 16, 2) LINK(1, 17, 3) LINK(2, 18, 3) LINK(3, 19, 3) LINK(4, 20, 3)
      : "+v"(acc)
      : "v"(w[0]), "v"(w[1]), "v"(w[2]), "v"(w[3]), "v"(a[0][0]), "v"(a[0][1]), "v"(a[0][2]), "v"(a[0][3]), "v"(a[1][0]), "v"(a[1][1]), "v"(a[1][2]),
        "v"(a[1][3]), "v"(a[2][0]), "v"(a[2][1]), "v"(a[2][2]), "v"(a[2][3]), "v"(a[3][0]), "v"(a[3][1]), "v"(a[3][2]), "v"(a[3][3]));
#undef LINK
  return acc;
}
template <bool GATED>
__global__ __launch_bounds__((GATED ? 6 : 5) * 64) void gemm_f32_few_kernel(const float* __restrict__ A, int lda, const float* __restrict__ W,
                                                                             const float* __restrict__ W2, const void* __restrict__ bias, int bias_dtype,
                                                                             void* __restrict__ out, int out_dtype, int ldo, int M, int N, int K,
                                                                             int epilogue, GateSpec gs) {
  using F = F32Few<GATED>;
  extern __shared__ __align__(1024) float lds[];  // [RING][BLOCKS][a block: 16 rows of W, of W2, 8 of A; 128 bytes a row]
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n0 = blockIdx.x * 16;
  const int turns = K / (F::BLOCKS * 32);
  if (wave >= F::NC) {
    const int me = wave - F::NC, row = lane >> 3, slot = lane & 7;
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) float*)lds;
    const float* at[F::LOADS];  // this lane's piece of each of the wave's loads of a turn
#pragma unroll
    for (int i = 0; i < F::LOADS; ++i) {
      const int u = me * F::LOADS + i, block = u / F::BLOCK_KB, part = u % F::BLOCK_KB;
      const int r = (part & 1) * 8 + row, k = block * 32 + (slot ^ ring_swz(part == 2 * F::NC ? row : r)) * 4;
      at[i] = (part == 2 * F::NC ? A + (size_t)min(row, M - 1) * lda : (part < 2 ? W : W2) + (size_t)min(n0 + r, N - 1) * K) + k;
    }
    auto issue = [&](int t, int place) {
#pragma unroll
      for (int i = 0; i < F::LOADS; ++i)
        load_to_lds_16(at[i] + (size_t)t * F::BLOCKS * 32, lds0 + (uint32_t)(place * F::TURN_KB + me * F::LOADS + i) * 1024u);
    };
#pragma unroll
    for (int t = 0; t < F::RING; ++t)
      if (t < turns) issue(t, t);
    int asked = min(F::RING, turns), place = 0;  // the place of turn t - 1
    for (int t = 0; t < turns; ++t) {
      switch (asked - 1 - t) {  // turns that may still be on their way
        case 3: wait_loads<(F::RING > 3 ? 3 : 0) * F::LOADS>(); break;
        case 2: wait_loads<2 * F::LOADS>(); break;
        case 1: wait_loads<1 * F::LOADS>(); break;
        default: wait_loads<0>();
      }
      __builtin_amdgcn_s_barrier();
      if (t == 0) continue;
      if (asked < turns) issue(asked++, place);
      if (++place == F::RING) place = 0;
    }
    if (GATED) __syncthreads();
    return;
  }
  const int r = lane >> 2, m = lane & 3, n = n0 + r;
  const bool mine = m < M && n < N;
  float prev = 0.f;
  if (epilogue == 1 && mine) prev = ((const float*)out)[(size_t)m * ldo + n];
  const float* wrow = lds + wave * 512 + r * 32;  // of a block
  const float* arow = lds + F::NC * 512 + m * 32;
  const int wswz = ring_swz(r), aswz = ring_swz(m);
  float acc = 0.f;
  for (int t0 = 0; t0 < turns; t0 += F::RING) {
#pragma unroll
    for (int place = 0; place < F::RING; ++place) {  // (each with its own addresses: an addition per read costs 7 %)
      if (t0 + place >= turns) break;
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      const int at = place * F::TURN_KB * 256;
      constexpr int CHUNKS = 2 * F::BLOCKS;  // of 16 k, each requested two ahead of its multiply-adds
      floatx4 w[3], a[3][4];
      auto read = [&](int i) {
        const int block = at + (i >> 1) * F::BLOCK_KB * 256, c = 4 * (i & 1);
        w[i % 3] = *(const floatx4*)(wrow + block + (((c + m) ^ wswz) << 2));
#pragma unroll
        for (int q = 0; q < 4; ++q) a[i % 3][q] = *(const floatx4*)(arow + block + (((c + q) ^ aswz) << 2));
      };
      read(0);
      read(1);
#pragma unroll
      for (int i = 0; i < CHUNKS; ++i) {
        if (i + 2 < CHUNKS) read(i + 2);
        __builtin_amdgcn_sched_barrier(0);
        acc = chain16(w[i % 3], a[i % 3], acc);
        __builtin_amdgcn_sched_barrier(0);
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the turn's last reads, before the barrier behind which it is filled again
    }
  }
  float up = 0.f;
  if (GATED) {
    __shared__ float meet[64];
    if (wave) meet[lane] = acc;
    __syncthreads();
    if (wave) return;
    up = meet[lane];
  }
  if (!mine) return;
  if (bias) acc += (bias_dtype == JLLM_BF16) ? ldf((const bf16_t*)bias, n) : ldf((const float*)bias, n);
  if (GATED) acc = gated<false>(acc, up, gs);
  const size_t o = (size_t)m * ldo + n;
  if (epilogue == 1)
    ((float*)out)[o] = prev + acc;
  else if (out_dtype == JLLM_BF16)
    stf((bf16_t*)out, o, acc);
  else
    stf((float*)out, o, acc);
}

#define GEMM_ROWS_MAX 16
#define GEMM_FEW_MAX 4

// Measured (fp32 operands, one product alone, against the vector-unit kernels that stood here): 2,048 x 4,096 x 4,096 1,029 ->
// 590 us (117 TFLOP/s; a library product reaches 154), 847 rows of N = 1,024 and K = 2,048 337 -> 51, K = 3,072 503 -> 73,
// 40 rows of the same 168 -> 20; up to 16 rows: N = 1,024 at K = 2,048 / 3,072 40 / 59 -> 12.5 / 17 us, N = 4,096 at K =
// 12,288 229 -> 71, the head of 151,936 x 1,024 218 -> 182 (3.4 TB/s).
//
// The tile is the one with the smallest estimated time: rounds of workgroups (one per compute unit) times the tile's
// products, the smaller tiles a little dearer for their share of loads. K cannot be cut (one accumulator per output), so
// where large tiles leave compute units idle only smaller ones fill them. The prices hold for both kernels: a full round of 64 x 64 takes
// 16.4 us per 1,024 k through the ring, one of 128 x 128 59.7.
struct F32Tile {
  int rows, cols;  // of the output
};
static int f32_tile(long M, long N, bool is_gated) {
  static const double price[3] = {1.0, 1.1, 1.4};  // 128 x 128, 64 x 64, 32 x 32 (gated: half the columns of the first two)
  const F32Tile plain[3] = {{128, 128}, {64, 64}, {32, 32}}, pairs[3] = {{128, 64}, {64, 32}, {32, 32}};
  int cus = jllm_compute_units();
  if (cus <= 0) cus = 256;
  int best = 0;
  double least = 0.0;
  for (int i = 0; i < 3; ++i) {
    const F32Tile t = is_gated ? pairs[i] : plain[i];
    const long rows = (M + t.rows - 1) / t.rows, groups = rows * ((N + t.cols - 1) / t.cols);
    const double cost = (double)((groups + cus - 1) / cus) * t.rows * t.cols * price[i];
    if (i == 0 || (cost < least && rows <= 65535)) best = i, least = cost;
  }
  return best;
}

extern "C" int jllm_f32_tile(int M, int N, int is_gated) { return f32_tile(M, N, is_gated != 0); }

struct F32Args {
  const void *A, *W, *W2, *bias;
  void* out;
  int lda, bias_dtype, out_dtype, ldo, M, N, K, epilogue;
  GateSpec gs;
};

template <typename TA, typename TW, bool GATED, int WM, int WN, int FM, int FN, int BK, bool WIDE>
static int launch_f32_tile(const F32Args& g, hipStream_t stream) {
  constexpr int TM = WM * FM * 16, TN = WN * FN * 16;
  constexpr size_t smem = (size_t)2 * (TM + (GATED ? 2 : 1) * TN) * BK * sizeof(float);
  static_assert(smem <= 65536, "no LDS beyond what a launch gets unasked");
  dim3 grid((g.N + TN - 1) / TN, (g.M + TM - 1) / TM);
  if (grid.y > 65535) JLLM_FAIL("gemm: M=%d is too large for this kernel", g.M);
  gemm_f32_tile_kernel<TA, TW, GATED, WM, WN, FM, FN, BK, WIDE><<<grid, WM * WN * 64, smem, stream>>>(
      (const TA*)g.A, g.lda, (const TW*)g.W, (const TW*)g.W2, g.bias, g.bias_dtype, g.out, g.out_dtype, g.ldo, g.M, g.N, g.K, g.epilogue, g.gs);
  return 0;
}

template <bool GATED, int WM, int WN, int FM, int FN, int RING>
static int launch_f32_ring(const F32Args& g, hipStream_t stream) {
  constexpr int TM = WM * FM * 16, TN = WN * FN * 16;
  constexpr size_t smem = (size_t)RING * (TM + (GATED ? 2 : 1) * TN) * 128;
  static bool configured = smem <= 65536;
  if (!configured) {
    if (hipFuncSetAttribute((const void*)gemm_f32_ring_kernel<GATED, WM, WN, FM, FN, RING>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem) != hipSuccess)
      JLLM_FAIL("gemm: cannot reserve %zu bytes of LDS", smem);
    configured = true;
  }
  dim3 grid((g.N + TN - 1) / TN, (g.M + TM - 1) / TM);
  if (grid.y > 65535) JLLM_FAIL("gemm: M=%d is too large for this kernel", g.M);
  gemm_f32_ring_kernel<GATED, WM, WN, FM, FN, RING><<<grid, WM * WN * 64, smem, stream>>>(
      (const float*)g.A, g.lda, (const float*)g.W, (const float*)g.W2, g.bias, g.bias_dtype, g.out, g.out_dtype, g.ldo, g.M, g.N, g.K, g.epilogue, g.gs);
  return 0;
}

template <bool GATED>
static int launch_f32_few(const F32Args& g, hipStream_t stream) {
  using F = F32Few<GATED>;
  static_assert(F::LDS + 64 * sizeof(float) <= 64 * 1024, "no launch needs leave for more");
  gemm_f32_few_kernel<GATED><<<(g.N + 15) / 16, F::THREADS, F::LDS, stream>>>((const float*)g.A, g.lda, (const float*)g.W, (const float*)g.W2, g.bias,
                                                                          g.bias_dtype, g.out, g.out_dtype, g.ldo, g.M, g.N, g.K, g.epilogue, g.gs);
  return 0;
}

template <typename TA, typename TW, bool WIDE>
static int launch_f32(const F32Args& g, hipStream_t stream) {
  if constexpr (WIDE && sizeof(TA) == 4 && sizeof(TW) == 4) {
    if (g.M <= GEMM_FEW_MAX && g.K % (F32Few<false>::BLOCKS * 32) == 0) return g.W2 ? launch_f32_few<true>(g, stream) : launch_f32_few<false>(g, stream);
  }
  if (g.M <= GEMM_ROWS_MAX) {
    dim3 grid((g.N + 15) / 16);
    if (g.W2)
      gemm_f32_rows_kernel<TA, TW, true, WIDE><<<grid, 320, 0, stream>>>((const TA*)g.A, g.lda, (const TW*)g.W, (const TW*)g.W2, g.bias,
                                                                         g.bias_dtype, g.out, g.out_dtype, g.ldo, g.M, g.N, g.K, g.epilogue, g.gs);
    else
      gemm_f32_rows_kernel<TA, TW, false, WIDE><<<grid, 256, 0, stream>>>((const TA*)g.A, g.lda, (const TW*)g.W, nullptr, g.bias,
                                                                         g.bias_dtype, g.out, g.out_dtype, g.ldo, g.M, g.N, g.K, g.epilogue, g.gs);
    return 0;
  }
  const int tile = f32_tile(g.M, g.N, g.W2 != nullptr);
  if constexpr (WIDE && sizeof(TA) == 4 && sizeof(TW) == 4) {
    // whole lines of 128 bytes of every row: the ring, faster at all of 17 .. 1,000 rows and eight shapes of products (by 6 to 25 %)
    if (g.K % 32 == 0) {
      if (g.W2)
        return tile == 0   ? launch_f32_ring<true, 2, 4, 4, 1, 3>(g, stream)
               : tile == 1 ? launch_f32_ring<true, 4, 2, 1, 1, 4>(g, stream)
                           : launch_f32_ring<true, 2, 2, 1, 1, 5>(g, stream);
      return tile == 0   ? launch_f32_ring<false, 2, 4, 4, 2, 3>(g, stream)
             : tile == 1 ? launch_f32_ring<false, 2, 4, 2, 1, 4>(g, stream)
                         : launch_f32_ring<false, 2, 2, 1, 1, 8>(g, stream);
    }
  }
  if (g.W2)
    return tile == 0   ? launch_f32_tile<TA, TW, true, 2, 4, 4, 1, 32, WIDE>(g, stream)
           : tile == 1 ? launch_f32_tile<TA, TW, true, 4, 2, 1, 1, 64, WIDE>(g, stream)
                       : launch_f32_tile<TA, TW, true, 2, 2, 1, 1, 64, WIDE>(g, stream);
  return tile == 0   ? launch_f32_tile<TA, TW, false, 2, 4, 4, 2, 32, WIDE>(g, stream)
         : tile == 1 ? launch_f32_tile<TA, TW, false, 2, 4, 2, 1, 64, WIDE>(g, stream)
                     : launch_f32_tile<TA, TW, false, 2, 2, 1, 1, 128, WIDE>(g, stream);
}

extern "C" int jllm_gemm_generic(const void* A, int a_dtype, int lda, const void* W, const void* W2, int w_dtype,
                                 const void* bias, int bias_dtype, void* out, int out_dtype, int ldo, int M, int N,
                                 int K, int epilogue, float gate_limit, hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (K <= 0) JLLM_FAIL("gemm: K=%d", K);
  if (lda < K || ldo < N) JLLM_FAIL("gemm: leading dimensions lda=%d K=%d ldo=%d N=%d", lda, K, ldo, N);
  JLLM_TAKE_GATE("gemm", epilogue, gate_limit, gs);
  if (epilogue < 0 || epilogue > 2) JLLM_FAIL("gemm: epilogue %d", epilogue);
  if ((epilogue == 2) != (W2 != nullptr)) JLLM_FAIL("gemm: the gated epilogue needs exactly two weight matrices");
  if (epilogue == 1 && out_dtype != JLLM_F32) JLLM_FAIL("gemm: the accumulate epilogue adds into fp32");
  const F32Args g = {A, W, W2, bias, out, lda, bias_dtype, out_dtype, ldo, M, N, K, epilogue, gs};
  // 16 bytes (fp32) or 8 bytes (bf16) at a time where every row of both operands starts on such a boundary and ends on one
  const size_t abytes = a_dtype == JLLM_F32 ? 16 : 8, wbytes = w_dtype == JLLM_F32 ? 16 : 8;
  const bool wide = (K & 3) == 0 && (lda & 3) == 0 && (uintptr_t)A % abytes == 0 && (uintptr_t)W % wbytes == 0 && (uintptr_t)W2 % wbytes == 0;
  int rc = 0;
  JLLM_DISPATCH_1(a_dtype, TA, {
    JLLM_DISPATCH_1(w_dtype, TW, { rc = wide ? launch_f32<TA, TW, true>(g, stream) : launch_f32<TA, TW, false>(g, stream); })
  })
  if (rc != 0) return rc;
  JLLM_CHECK_LAUNCH("gemm_generic");
  return 0;
}
