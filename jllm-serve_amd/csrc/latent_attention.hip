// Latent attention on the matrix cores, bf16: one kernel for single decoded rows, one for portions of prompts.
//
// All heads of a row attend over the same cached rows (Dk = R + Dr numbers per position, the first R of which are also
// the values), so the query vectors of many heads (and rows) share every key they read. A workgroup takes up to 64 query
// vectors. It walks the keys they can see in blocks of 64 aligned to absolute positions, and stages each block once in LDS as
// it lies in the cache (two buffers take turns: the next block travels while this one is multiplied). Per 16 keys a wave computes
//   S^T = K . Q^T   (MFMA 16x16x32; K fragments from LDS, Q^T in registers): a lane then holds four keys' scores of
//                   ONE query vector, so masks (causal and window, per query vector), maximum and sum need only two
//                   shuffles over the lane groups;
//   O^T += V^T . P^T: those probabilities, packed to bf16, are the B operand, and V^T is read from the staged block
//                   with the transposing LDS load.
// The running maximum moves only when it grows by more than 8 (probabilities stay below e^8, exact in fp32 sums).
// exp(sink) of the query vector's head joins the denominator at the end. Scores, softmax and sums are fp32.
//
// The runs come from the step's plan: (request, first row, rows <= 16, -) per tile; positions are read per row.
//
// Single rows: eight waves, of which w and w + 4 own the same 16 query vectors (heads) and both compute their scores and
// softmax, but each keeps only one half of the latent's accumulators (a 512-wide latent is 128 registers per lane).
// Steps with few workgroups cut every row's keys into absolute ranges of `split` keys over
// gridDim.z: a workgroup then leaves maximum, sum and unnormalised sums per query vector, and a second kernel merges
// the ranges in ascending order, adds the sink and normalises.
#include <math.h>

#include "common.h"
#include "mfma.h"

#define LM_WAVES 8
#define LM_QW 4  // waves with query vectors of their own; waves 4..7 repeat them for the other half of the latent
#define LM_KEYS 64
#define LM_TILE_ROWS 16
#define LM_AHEAD 4  // fragments of keys requested ahead of the multiplies
#define LM_PS (LM_KEYS + 8)  // elements between two query vectors' probabilities

__device__ __forceinline__ float lm_exp_diff(float a, float b) { return a == -INFINITY ? 0.f : __expf(a - b); }

// RT: 16-dim blocks of the latent the accumulators hold at most; DKS: 32-dim steps of a key row at most
// WHOLE: the sizes are exactly those, and nothing in the loops is conditional on them: a step behind a condition waits for its own LDS
// read, eighteen times a score and sixteen a sum. Single rows of 512 + 64 entries, us with the merge, before / so (a workgroup is a chain
// of blocks of 64 keys, 2.8 -> 1.9 us each at 16 heads, 7.3 -> 4.0 at 32): 8 rows of 16 heads and a window of 1,024 in ranges of 128 keys
// 20.2 / 16.2, in ranges of 64 18.1 / 14.7; 32 heads 24.4 / 18.2 and 18.1 / 14.7; 24 rows of 32 heads and 2,000 keys in ranges of 384 58 / 39.
// Sizes in between keep the conditions: padded to these they would multiply up to three times their entries and hold a compute unit's LDS.
template <int RT, int DKS, bool WHOLE>
__global__ __launch_bounds__(LM_WAVES * 64) void latent_attention_mfma_kernel(
    const bf16_t* __restrict__ qa, int ldq, bf16_t* __restrict__ out, int ldo, const bf16_t* __restrict__ cache,
    const int* __restrict__ block_table, int max_blocks, const int* __restrict__ tiles,
    const int* __restrict__ positions, int H, int R, int Dk, int page_size, int window, float scale,
    const float* __restrict__ sink, int HB, int LD, int split, float* __restrict__ part) {
  extern __shared__ __align__(16) unsigned char lm_smem[];
  bf16_t* Ks = (bf16_t*)lm_smem;  // [2][LM_KEYS][LD]
  const int tile = blockIdx.x;
  const int req = tiles[4 * tile], row = tiles[4 * tile + 1];
  const int hb = blockIdx.y;
  int ke = positions[row];
  int kb = window > 0 ? max(0, ke + 1 - window) : 0;
  if (split > 0) {  // this workgroup's range of the row's keys
    const int s0 = kb / split + (int)blockIdx.z;
    kb = max(kb, s0 * split);
    ke = min(ke, s0 * split + split - 1);
    if (kb > ke) return;
  }
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int sub = lane & 15, q4 = lane >> 4;
  // At most 16 heads are 16 query vectors, one wave's worth: then all four waves take the same query vectors and
  // every fourth group of 16 keys each, and merge at the end in the order of the waves.
  const bool kpar = HB <= 16;
  const int qwave = wave & (LM_QW - 1), rhalf = wave / LM_QW;
  const int v = kpar ? sub : qwave * 16 + sub;
  const int my_h = hb * HB + v;
  const bool live = v < HB && my_h < H;
  const bool wave_live = kpar || qwave * 16 < HB;  // (a wave without a live query vector only helps to load)
  const int dks = WHOLE ? DKS : (Dk + 31) >> 5, r16 = WHOLE ? RT : R >> 4;
  constexpr int RTH = (RT + 1) / 2;  // accumulators of one wave: its half of the latent's 16-dim blocks
  static_assert(!WHOLE || (RT % 2 == 0 && DKS % 2 == 0), "two equal halves of the latent, and a row in loads of 64 entries");
  const int j_lo = rhalf ? (r16 + 1) / 2 : 0, nj = WHOLE ? RTH : rhalf ? r16 - (r16 + 1) / 2 : (r16 + 1) / 2;
  const int psh = __builtin_ctz(page_size);
  const int* tbl = block_table + (size_t)req * max_blocks;

  u32x4 qf[DKS];
  {
    const bf16_t* qrow = qa + (size_t)row * ldq + (size_t)min(my_h, H - 1) * Dk;
#pragma unroll
    for (int j = 0; j < DKS; ++j) {
      const int d = 32 * j + 8 * q4;
      qf[j] = (WHOLE || (live && j < dks && d < Dk)) ? *(const u32x4*)(qrow + d) : u32x4{0u, 0u, 0u, 0u};  // (WHOLE: another head's where not live, unused)
    }
  }
  floatx4 acc[RTH];
#pragma unroll
  for (int j = 0; j < RTH; ++j) acc[j] = floatx4{0.f, 0.f, 0.f, 0.f};
  float m1 = -INFINITY, l1 = 0.f;
  // A block of 64 keys goes global -> registers -> LDS. All of a thread's pieces are requested together (first their
  // table entries, then the rows: two latencies a block, not two per piece), and the next block's are requested before
  // this block is multiplied, into the other of two LDS buffers: one barrier per block.
  // eight threads to a key row (512 threads, 64 rows): a thread's pieces are 16 bytes at (tid % 8) * 16 + 128 i of its
  // row: one table entry and one address per block
  constexpr int CPT = (DKS + 1) / 2;
  static_assert(LM_WAVES * 64 == 8 * LM_KEYS, "eight threads stage a key row");
  uint4 staged[CPT];
  const int srow = threadIdx.x >> 3, scol = (threadIdx.x & 7) * 8;
  auto fetch = [&](int blk) {
    const int key = min(max(blk * LM_KEYS + srow, kb), ke);  // a key outside the range is masked below and reads one inside it
    const bf16_t* src = cache + ((((size_t)tbl[key >> psh]) << psh) + (key & (page_size - 1))) * Dk + scol;
#pragma unroll
    for (int i = 0; i < CPT; ++i) staged[i] = (WHOLE || scol + 64 * i < Dk) ? *(const uint4*)(src + 64 * i) : uint4{0u, 0u, 0u, 0u};
  };
  auto put = [&](bf16_t* buf) {
    bf16_t* dst = buf + srow * LD + scol;
#pragma unroll
    for (int i = 0; i < CPT; ++i)
      if (WHOLE || scol + 64 * i < dks * 32) *(uint4*)(dst + 64 * i) = staged[i];
  };
  const int blk_last = ke >> 6;
  int cur = 0;
  fetch(kb >> 6);
  put(Ks);
  __syncthreads();
  for (int blk = kb >> 6; blk <= blk_last; ++blk) {
    const int c0 = blk * LM_KEYS;
    const bf16_t* Kb = Ks + (size_t)cur * LM_KEYS * LD;
    if (blk < blk_last) fetch(blk + 1);
    if (wave_live) {
#pragma unroll 1
      for (int st = 0; st < LM_KEYS / 16; ++st) {
        const int k0 = c0 + st * 16;
        if (k0 + 15 < kb || k0 > ke) continue;  // none of these keys is this workgroup's
        if (kpar && st != qwave) continue;           // another wave's keys
        floatx4 sc = floatx4{0.f, 0.f, 0.f, 0.f}, sc2 = floatx4{0.f, 0.f, 0.f, 0.f};  // two chains of dependent MFMAs
        const bf16_t* krow = Kb + (st * 16 + sub) * LD + 8 * q4;
#pragma unroll
        for (int j = 0; j < DKS; j += 2) {
          if (j < dks) sc = mfma16(*(const u32x4*)(krow + 32 * j), qf[j], sc);
          if (j + 1 < DKS && j + 1 < dks) sc2 = mfma16(*(const u32x4*)(krow + 32 * (j + 1)), qf[j + 1 < DKS ? j + 1 : j], sc2);
        }
        sc += sc2;
        float z[4];
        float mx = -INFINITY;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int key = k0 + 4 * q4 + i;
          z[i] = (live && key >= kb && key <= ke) ? sc[i] * scale : -INFINITY;
          mx = fmaxf(mx, z[i]);
        }
        mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
        mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
        if (mx > m1 + 8.0f) {  // also the first visible key (m1 = -inf)
          const float alpha = lm_exp_diff(m1, mx);
          l1 *= alpha;
#pragma unroll
          for (int j = 0; j < RTH; ++j) acc[j] *= alpha;
          m1 = mx;
        }
        float p[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          p[i] = lm_exp_diff(z[i], m1);
          l1 += p[i];
        }
        const u32x2 pb = u32x2{pack_bf16(p[0], p[1]), pack_bf16(p[2], p[3])};
        const bf16_t* v_tr = Kb + (st * 16 + 4 * q4 + (sub >> 2)) * LD + 4 * (sub & 3);
#pragma unroll
        for (int j = 0; j < RTH; ++j)
          if (j < nj) acc[j] = mfma16k16(lds_read_tr16(v_tr + 16 * (j_lo + j)), pb, acc[j]);
      }
    }
    if (blk < blk_last) put(Ks + (size_t)(cur ^ 1) * LM_KEYS * LD);
    __syncthreads();  // the other buffer is whole, and everyone is done with this one
    cur ^= 1;
  }
  l1 += __shfl_xor(l1, 16, 64);
  l1 += __shfl_xor(l1, 32, 64);
  if (kpar) {  // the loop's last barrier has passed: the key buffers now carry the merge
    constexpr int MS = 2 + 4 * RTH;
    float* mrg = (float*)lm_smem + (size_t)rhalf * (LM_QW - 1) * 64 * MS;  // [2][LM_QW - 1][64][MS]
    if (qwave > 0) {
      float* d = mrg + (size_t)((qwave - 1) * 64 + lane) * MS;
      d[0] = m1, d[1] = l1;
#pragma unroll
      for (int j = 0; j < RTH; ++j)
        if (j < nj) {
#pragma unroll
          for (int i = 0; i < 4; ++i) d[2 + 4 * j + i] = acc[j][i];
        }
    }
    __syncthreads();
    if (qwave > 0) return;
#pragma unroll 1
    for (int w = 0; w < LM_QW - 1; ++w) {
      const float* src = mrg + (size_t)(w * 64 + lane) * MS;
      const float om = src[0], ol = src[1];
      const float mn = fmaxf(m1, om);
      const float a = lm_exp_diff(m1, mn), b = lm_exp_diff(om, mn);
      l1 = l1 * a + ol * b;
#pragma unroll
      for (int j = 0; j < RTH; ++j)
        if (j < nj) {
#pragma unroll
          for (int i = 0; i < 4; ++i) acc[j][i] = acc[j][i] * a + src[2 + 4 * j + i] * b;
        }
      m1 = mn;
    }
  }
  if (!live) return;
  if (split > 0) {
    float* dst = part + (((size_t)row * H + my_h) * gridDim.z + blockIdx.z) * (R + 4);  // R sums, maximum, sum
    if (q4 == 0 && rhalf == 0) dst[R] = m1, dst[R + 1] = l1;
#pragma unroll
    for (int j = 0; j < RTH; ++j)
      if (j < nj) *(floatx4*)(dst + 16 * (j_lo + j) + 4 * q4) = acc[j];
    return;
  }
  float ca = 1.0f;
  if (sink) {
    const float sk = sink[my_h];
    const float mn = fmaxf(m1, sk);
    ca = lm_exp_diff(m1, mn);
    l1 = l1 * ca + __expf(sk - mn);
  }
  const float inv = ca / l1;
  bf16_t* o = out + (size_t)row * ldo + (size_t)my_h * R + 4 * q4;
#pragma unroll
  for (int j = 0; j < RTH; ++j)
    if (j < nj)
      *(u32x2*)(o + 16 * (j_lo + j)) = u32x2{pack_bf16(acc[j][0] * inv, acc[j][1] * inv), pack_bf16(acc[j][2] * inv, acc[j][3] * inv)};
}

// Runs of several rows (portions of prompts). A workgroup takes 64 query vectors of one run (HB heads x 64 / HB rows) and
// walks the keys they can see in blocks of 64 as the kernel above, but no product is computed twice: wave w computes the
// scores of 16 query vectors (w % 4) with 32 of a block's keys (w / 4), its queries in registers; the waves agree on the
// block's maxima over LDS, leave their probabilities there as bf16, and wave w then sums all 64 query vectors' values over
// an eighth of the latent. A V^T fragment so serves four products and only the scores' K fragments one. What bounds
// it are those: 288 KB of LDS reads a block of 64 keys of 576 entries. Two barriers a block: the scores of a block
// follow the sums of the one before without one. Nothing in the loops is conditional on sizes (a conditional step waits for
// its own LDS reads): rows are staged with zeros up to DKS steps of 32.
//
// A row has the bits that the kernel above gives it: scores in two chains, the running maximum and the denominator
// moved 16 keys at a time (the waves of a block's first 32 keys hand the denominators to those of the second), 32 keys of
// values in one product (the matrix core adds the first 16 and then the others, as two products of 16 do), a row
// alone with at most 16 heads in four sums, one for every fourth 16 keys. A key that a row does not see is multiplied by
// 0, which an infinite value would not survive: a result that is no finite number is computed again from its own keys.
//
// 16 heads, 512 + 64 entries, against the kernel above, which took these runs too and computed every score twice: prompts
// of 300 to 1,211 rows (3,611 in all) 400 -> 186 us, 487 rows 73 -> 36, a portion of 30 rows and three single rows of 1,500 keys
// 85 -> 73, 2,048 rows with a window of 512 165 -> 88. With scores in one chain and maxima moved 64 keys at a time,
// in other bits, 168, 32, 78 and 78.
template <int NJ, int DKS>  // NJ: 16-dim blocks of the latent per wave at most (8 NJ >= R / 16); DKS as above
__global__ __launch_bounds__(LM_WAVES * 64) void latent_attention_rows_kernel(
    const bf16_t* __restrict__ qa, int ldq, bf16_t* __restrict__ out, int ldo, const bf16_t* __restrict__ cache,
    const int* __restrict__ block_table, int max_blocks, const int* __restrict__ tiles, const int* __restrict__ positions,
    int H, int R, int Dk, int page_size, int window, float scale, const float* __restrict__ sink, int HB, int n_hb) {
  constexpr int LD = DKS * 32 + 16;          // elements between two keys' rows in LDS (16 mod 64: see the launch)
  extern __shared__ __align__(16) unsigned char lm_smem[];
  bf16_t* Ks = (bf16_t*)lm_smem;             // [2][LM_KEYS][LD]
  bf16_t* Ps = Ks + (size_t)2 * LM_KEYS * LD;  // [64 query vectors][LM_PS]: a block's probabilities
  float* mxs = (float*)(Ps + 64 * LM_PS);    // [4][64]: the maxima over the block's four 16 keys; at the end the results' factors
  floatx4* als = (floatx4*)(mxs + 256);      // [64]: the factors of what was summed before each of them
  float* den = (float*)(als + 64);           // [4][64]: a lane's part of its denominator, between the waves of a block's halves
  const int tile = blockIdx.x;
  const int req = tiles[4 * tile], row0 = tiles[4 * tile + 1], rows = tiles[4 * tile + 2];
  const int RW = 64 / HB;
  const int hb = blockIdx.y % n_hb, r_lo = blockIdx.y / n_hb * RW;
  if (r_lo >= rows) return;
  const int r_hi = min(rows, r_lo + RW) - 1;
  const int p_lo = positions[row0 + r_lo];
  const int kb = window > 0 ? max(0, p_lo + 1 - window) : 0, ke = p_lo + (r_hi - r_lo);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int sub = lane & 15, q4 = lane >> 4;
  const int qs = wave & 3, kh = wave >> 2;
  const bool alone = r_hi == r_lo && HB <= 16;  // the four groups of 16 query vectors are the same ones over every fourth 16 keys
  const int v = qs * 16 + sub;  // this lane's query vector of the scores
  const int my_r = r_lo + (alone ? sub : v) / HB, my_h = hb * HB + (alone ? sub : v) % HB;
  const bool live = my_r <= r_hi && my_h < H;
  const int my_pos = p_lo + (my_r - r_lo);
  const int my_first = !live ? 0x7fffffff : window > 0 ? max(0, my_pos + 1 - window) : 0;  // (dead: sees no key)
  const int n_q = alone ? 4 : min(4, ((r_hi - r_lo + 1) * HB + 15) >> 4);  // groups of 16 query vectors with a row
  const int last_first = window > 0 ? max(0, ke + 1 - window) : 0;         // from here on to p_lo all rows see a key
  const int j_lo = wave * NJ, nj = min(NJ, (R >> 4) - j_lo);
  const int psh = __builtin_ctz(page_size);
  const int* tbl = block_table + (size_t)req * max_blocks;

  u32x4 qf[DKS];
  {
    const bf16_t* qrow = qa + (size_t)(row0 + min(my_r, r_hi)) * ldq + (size_t)min(my_h, H - 1) * Dk;
#pragma unroll
    for (int j = 0; j < DKS; ++j) {
      const int d = 32 * j + 8 * q4;
      qf[j] = (live && d < Dk) ? *(const u32x4*)(qrow + d) : u32x4{0u, 0u, 0u, 0u};
    }
  }
  floatx4 acc[4][NJ];
#pragma unroll
  for (int q = 0; q < 4; ++q)
#pragma unroll
    for (int j = 0; j < NJ; ++j) acc[q][j] = floatx4{0.f, 0.f, 0.f, 0.f};
  float m1 = -INFINITY, l1 = 0.f;
  if (threadIdx.x < 64) als[threadIdx.x] = floatx4{1.f, 1.f, 1.f, 1.f};  // (of groups without a row they stay so)
  // keys travel as above (eight threads to a key row, the next block's in registers while this one is multiplied); a
  // block's page is looked up a block before its rows are requested
  constexpr int CPT = (DKS + 1) / 2;
  uint4 staged[CPT];
  const int srow = threadIdx.x >> 3, scol = (threadIdx.x & 7) * 8;
  const int blk_last = ke >> 6;
  int blk = kb >> 6;
  auto key_of = [&](int b) { return min(max(b * LM_KEYS + srow, kb), ke); };  // (a key outside the range is masked and reads one inside it)
  int page = tbl[key_of(blk) >> psh];
  auto fetch = [&](int b) {
    const bf16_t* src = cache + ((((size_t)page) << psh) + (key_of(b) & (page_size - 1))) * Dk;
    int left = Dk - scol;
    asm volatile("" : "+v"(left));
#pragma unroll
    for (int i = 0; i < CPT; ++i) staged[i] = *(const uint4*)(src + (64 * i < left ? scol + 64 * i : 0));
    page = tbl[key_of(b + 1) >> psh];
  };
  auto put = [&](bf16_t* buf) {
    bf16_t* dst = buf + srow * LD + scol;
    int left = Dk - scol;  // (compared per block: the nine results would be held over the loop)
    asm volatile("" : "+v"(left));
#pragma unroll
    for (int i = 0; i < CPT; ++i)
      *(uint4*)(dst + 64 * i) = 64 * i < left ? staged[i] : uint4{0u, 0u, 0u, 0u};
  };
  fetch(blk);
  put(Ks);
  __syncthreads();
  for (int cur = 0; blk <= blk_last; ++blk, cur ^= 1) {
    const int c0 = blk * LM_KEYS;
    const bf16_t* Kb = Ks + (size_t)cur * LM_KEYS * LD;
    if (blk < blk_last) fetch(blk + 1);
    float z[8];
    if (alone) {  // the waves of one half of the block have nothing to do, the others one 16 keys
#pragma unroll
      for (int i = 0; i < 8; ++i) z[i] = -INFINITY;
      float mx = -INFINITY;
      if (kh == qs >> 1) {
        floatx4 sc[2];
        sc[0] = sc[1] = floatx4{0.f, 0.f, 0.f, 0.f};
        const bf16_t* krow = Kb + (qs * 16 + sub) * LD + 8 * q4;
        u32x4 kf[LM_AHEAD + 1];
#pragma unroll
        for (int j = 0; j < DKS + LM_AHEAD; ++j) {
          if (j < DKS) kf[j % (LM_AHEAD + 1)] = *(const u32x4*)(krow + 32 * j);
          if (j >= LM_AHEAD) sc[(j - LM_AHEAD) & 1] = mfma16(kf[(j - LM_AHEAD) % (LM_AHEAD + 1)], qf[j - LM_AHEAD], sc[(j - LM_AHEAD) & 1]);
          __builtin_amdgcn_sched_barrier(0);
        }
        const floatx4 s = sc[0] + sc[1];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int key = c0 + qs * 16 + 4 * q4 + i;
          const float x = (key >= my_first && key <= my_pos) ? s[i] * scale : -INFINITY;
          if (qs & 1)
            z[4 + i] = x;
          else
            z[i] = x;
          mx = fmaxf(mx, x);
        }
        mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
        mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
      }
#pragma unroll
      for (int g = 0; g < 2; ++g)
        if (q4 == 0) mxs[(2 * kh + g) * 64 + v] = 2 * kh + g == qs ? mx : -INFINITY;
    } else if (qs < n_q) {
      floatx4 sc[2][2];  // two chains for each of the wave's two 16 keys
#pragma unroll
      for (int i = 0; i < 4; ++i) sc[i >> 1][i & 1] = floatx4{0.f, 0.f, 0.f, 0.f};
      const bf16_t* krow = Kb + (kh * 32 + sub) * LD + 8 * q4;
      u32x4 kf[LM_AHEAD + 1];
#pragma unroll
      for (int j = 0; j < 2 * DKS + LM_AHEAD; ++j) {  // fragments LM_AHEAD steps ahead of the multiplies, no more: registers
        if (j < 2 * DKS) kf[j % (LM_AHEAD + 1)] = *(const u32x4*)(krow + j / DKS * 16 * LD + 32 * (j % DKS));
        if (j >= LM_AHEAD) {
          const int m = j - LM_AHEAD, d = m % DKS;
          sc[m / DKS][d & 1] = mfma16(kf[m % (LM_AHEAD + 1)], qf[d], sc[m / DKS][d & 1]);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int g = 0; g < 2; ++g) {
        const floatx4 s = sc[g][0] + sc[g][1];
        float mx = -INFINITY;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int key = c0 + kh * 32 + g * 16 + 4 * q4 + i;
          z[4 * g + i] = (key >= my_first && key <= my_pos) ? s[i] * scale : -INFINITY;
          mx = fmaxf(mx, z[4 * g + i]);
        }
        mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
        mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
        if (q4 == 0) mxs[(2 * kh + g) * 64 + v] = mx;
      }
    }
    __syncthreads();  // the maxima are there, and everyone is done with the last block's probabilities and keys
    if (blk < blk_last) put(Ks + (size_t)(cur ^ 1) * LM_KEYS * LD);
    float al[4];
    if (qs < n_q) {
      float m[4];
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const float mx = mxs[g * 64 + v];
        al[g] = 1.0f;
        if (mx > m1 + 8.0f) {  // also the first visible key (m1 = -inf: nothing was summed yet)
          al[g] = m1 == -INFINITY ? 1.0f : __expf(m1 - mx);
          m1 = mx;
        }
        m[g] = m1;
      }
      if (kh == 0 && q4 == 0) als[v] = floatx4{al[0], al[1], al[2], al[3]};
#pragma unroll
      for (int i = 0; i < 8; ++i) z[i] = lm_exp_diff(z[i], kh ? m[2 + (i >> 2)] : m[i >> 2]);
      if (kh == 0) {
        if (blk > (kb >> 6)) l1 = den[qs * 64 + lane];
        l1 *= al[0];
        l1 += z[0], l1 += z[1], l1 += z[2], l1 += z[3];
        l1 *= al[1];
        l1 += z[4], l1 += z[5], l1 += z[6], l1 += z[7];
        den[qs * 64 + lane] = l1;
      }
      bf16_t* p = Ps + v * LM_PS + kh * 32 + 4 * q4;
      *(u32x2*)p = u32x2{pack_bf16(z[0], z[1]), pack_bf16(z[2], z[3])};
      *(u32x2*)(p + 16) = u32x2{pack_bf16(z[4], z[5]), pack_bf16(z[6], z[7])};
    }
    __syncthreads();  // the probabilities and the next block's keys are there
    if (kh == 1 && qs < n_q) {
      l1 = den[qs * 64 + lane];
      const floatx4 f = als[v];
      l1 *= f[2];
      l1 += z[0], l1 += z[1], l1 += z[2], l1 += z[3];
      l1 *= f[3];
      l1 += z[4], l1 += z[5], l1 += z[6], l1 += z[7];
      den[qs * 64 + lane] = l1;
    }
    const floatx4 moved = als[lane];  // lane u: of query vector u; the waves come to the same answer
    int starts = 0;                   // the groups of 16 keys in front of which some maximum moved
    if (__any(moved[0] != 1.0f || moved[1] != 1.0f || moved[2] != 1.0f || moved[3] != 1.0f)) {
#pragma unroll
      for (int g = 0; g < 4; ++g) starts |= __any(moved[g] != 1.0f) ? 1 << g : 0;
    }
    const bf16_t* v_tr = Kb + (8 * q4 + (sub >> 2)) * LD + 4 * (sub & 3) + 16 * j_lo;
    const bf16_t* prow = Ps + sub * LM_PS + 8 * q4;
    auto values = [&](u32x4 (&vf)[NJ], int half) {
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        const u32x2 a = lds_read_tr16(v_tr + half * 32 * LD + 16 * j), b = lds_read_tr16(v_tr + (half * 32 + 4) * LD + 16 * j);
        vf[j] = u32x4{a[0], a[1], b[0], b[1]};
      }
    };
    // the whole block at once or, where a maximum moved inside it (rare), the keys up to there first: the others'
    // probabilities count as zeros
#pragma unroll 1
    for (int g = 0, next; g < 4; g = next) {
      next = __builtin_ctz((starts >> (g + 1) << (g + 1)) | 16);
      uint32_t keep[2] = {~0u, ~0u};
      if (starts) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const float a = ((const float*)als)[(q * 16 + sub) * 4 + g];
#pragma unroll
          for (int j = 0; j < NJ; ++j) acc[q][j] *= a;
        }
#pragma unroll
        for (int half = 0; half < 2; ++half) keep[half] = 2 * half + (q4 >> 1) >= g && 2 * half + (q4 >> 1) < next ? ~0u : 0u;
      }
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        u32x4 vf[NJ];
        values(vf, half);
        const u32x4 p0 = *(const u32x4*)(prow + half * 32) & keep[half];
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[0][j] = mfma16(vf[j], p0, acc[0][j]);
        if (n_q > 1) {
#pragma unroll
          for (int q = 1; q < 4; ++q) {
            const u32x4 pf = *(const u32x4*)(prow + q * 16 * LM_PS + half * 32) & keep[half];
#pragma unroll
            for (int j = 0; j < NJ; ++j) acc[q][j] = mfma16(vf[j], pf, acc[q][j]);
          }
        }
      }
    }
  }
  // the denominators lie with the waves of the blocks' second halves
  l1 += __shfl_xor(l1, 16, 64);
  l1 += __shfl_xor(l1, 32, 64);
  auto factor = [&](float m, float l, int h) {
    float ca = 1.0f;
    if (sink) {
      const float sk = sink[h];
      const float mn = fmaxf(m, sk);
      ca = lm_exp_diff(m, mn);
      l = l * ca + __expf(sk - mn);
    }
    return ca / l;
  };
  if (kh == 1 && q4 == 0) {
    if (alone)
      mxs[v] = m1, mxs[64 + v] = l1;
    else if (live)
      mxs[v] = factor(m1, l1, my_h);
  }
  __syncthreads();
  // one query vector's sums over this wave's part of the latent, key by key
  auto again = [&](int r, int h) {
    const bf16_t* qrow = qa + (size_t)(row0 + r) * ldq + (size_t)h * Dk;
    const int pos = p_lo + (r - r_lo), first = window > 0 ? max(0, pos + 1 - window) : 0;
    const int dim = 16 * j_lo + lane;
    float m = -INFINITY, l = 0.f, o = 0.f;
    for (int k0 = first; k0 <= pos; k0 += 64) {
      const int key = min(k0 + lane, pos);
      const int at = (tbl[key >> psh] << psh) + (key & (page_size - 1));
      float d = 0.f;
      for (int i = 0; i < Dk; ++i) d = fmaf(ldf(qrow, i), ldf(cache + (size_t)at * Dk, i), d);
      const float z1 = k0 + lane <= pos ? d * scale : -INFINITY;
      const float mn = fmaxf(m, wave_max(z1)), a = lm_exp_diff(m, mn);
      const float p = lm_exp_diff(z1, mn);
      l = l * a + wave_sum(p);
      o *= a;
      m = mn;
      for (int k = 0; k < 64 && k0 + k <= pos; ++k) {
        const bf16_t* row = cache + (size_t)__shfl(at, k, 64) * Dk;
        o = fmaf(__shfl(p, k, 64), lane < 16 * nj ? ldf(row, dim) : 0.f, o);
      }
    }
    if (lane < 16 * nj) stf(out + (size_t)(row0 + r) * ldo, (size_t)h * R + dim, o * factor(m, l, h));
  };
  if (alone) {  // the four sums, in order
    float m = mxs[sub], l = mxs[64 + sub];
#pragma unroll
    for (int w = 1; w < 4; ++w) {
      const float om = mxs[16 * w + sub], ol = mxs[64 + 16 * w + sub];
      const float mn = fmaxf(m, om);
      const float a = lm_exp_diff(m, mn), b = lm_exp_diff(om, mn);
      l = l * a + ol * b;
#pragma unroll
      for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[0][j][i] = acc[0][j][i] * a + acc[w][j][i] * b;
      m = mn;
    }
    if (sub < HB && hb * HB + sub < H) mxs[128 + sub] = factor(m, l, hb * HB + sub);  // (every wave and lane group the same)
  }
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int u = q * 16 + sub, row = r_lo + u / HB, h = hb * HB + u % HB;
    const bool stored = (alone ? u < HB : row <= r_hi) && h < H;
    const float inv = mxs[alone ? 128 + sub : u];
    bf16_t* o = out + (size_t)(row0 + row) * ldo + (size_t)h * R + 16 * j_lo + 4 * q4;
    bool odd = false;
#pragma unroll
    for (int j = 0; j < NJ; ++j)
      if (stored && j < nj) {
        const floatx4 x = acc[q][j] * inv;
#pragma unroll
        for (int i = 0; i < 4; ++i) odd = odd || !(fabsf(x[i]) < INFINITY);
        *(u32x2*)(o + 16 * j) = u32x2{pack_bf16(x[0], x[1]), pack_bf16(x[2], x[3])};
      }
    const uint64_t lanes = __ballot(odd);
    uint32_t again_for = (uint32_t)(lanes | lanes >> 16 | lanes >> 32 | lanes >> 48) & 0xffffu;
    for (; again_for; again_for &= again_for - 1) {
      const int w = q * 16 + __builtin_ctz(again_for);
      again(r_lo + w / HB, hb * HB + w % HB);
    }
  }
}

// merges the key ranges of one (row, head); four waves per (row, head), a thread owns dims tid and tid + 256. Lane z of
// every wave first takes range z's maximum and sum (all ranges at once: n_z <= 64), the wave agrees on the overall
// maximum and every range's weight, and then the weighted sums are added in ascending order of the ranges with eight
// ranges' loads in flight. 8 rows of 16 heads of 512 in 17 ranges 7.7 -> 4.7 us since no branch stands around a load.
__global__ __launch_bounds__(256) void latent_attention_merge_kernel(const float* __restrict__ part, const int* __restrict__ positions,
                                                                   int H, int R, int window, int split, int n_z,
                                                                   const float* __restrict__ sink, bf16_t* __restrict__ out,
                                                                   int ldo) {
  const int t = blockIdx.x, h = blockIdx.y, lane = threadIdx.x & 63;
  const int pos = positions[t];
  const int first = window > 0 ? max(0, pos + 1 - window) : 0;
  const int s0 = first / split;
  const int n_valid = min(n_z, pos / split - s0 + 1);  // the ranges that hold keys of this row
  const float* base = part + ((size_t)t * H + h) * n_z * (R + 4);
  // no branch around a load (the compiler would wait for everything behind one): dims beyond R are the last one again, ranges
  // beyond n_valid the last one, neither is used
  const int dd[2] = {min((int)threadIdx.x, R - 1), min((int)threadIdx.x + 256, R - 1)};
  float pv[8][2];
  auto request = [&](int z0) {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float* src = base + (size_t)min(z0 + j, n_valid - 1) * (R + 4);
#pragma unroll
      for (int a = 0; a < 2; ++a) pv[j][a] = src[dd[a]];
    }
  };
  const float* mine = base + (size_t)min(lane, n_valid - 1) * (R + 4) + R;
  const float pm_there = mine[0], pl_there = mine[1];
  request(0);
  const float pm = lane < n_valid ? pm_there : -INFINITY, pl = lane < n_valid ? pl_there : 0.f;
  float m = wave_max(pm);
  const float sk = sink ? sink[h] : -INFINITY;
  m = fmaxf(m, sk);
  const float wz = lm_exp_diff(pm, m);
  float l = wave_sum(pl * wz) + (sink ? __expf(sk - m) : 0.f);
  float acc[2] = {0.f, 0.f};  // R <= 512
  for (int z0 = 0; z0 < n_valid; z0 += 8) {
    if (z0 > 0) request(z0);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float w = __shfl(wz, min(z0 + j, 63), 64);
      if (z0 + j < n_valid) {
#pragma unroll
        for (int a = 0; a < 2; ++a) acc[a] = fmaf(pv[j][a], w, acc[a]);
      }
    }
  }
  const float inv = 1.0f / l;
#pragma unroll
  for (int a = 0; a < 2; ++a) {
    const int d = threadIdx.x + 256 * a;
    if (d < R) stf(out + (size_t)t * ldo + (size_t)h * R, d, acc[a] * inv);
  }
}

template <int RT, int DKS, bool WHOLE>
static int lm_launch_as(dim3 grid, size_t smem, hipStream_t stream, const void* qa, int ldq, void* out, int ldo, const void* cache,
                     const int* block_table, int max_blocks, const int* tiles, const int* positions, int H, int R, int Dk,
                     int page_size, int window, float scale, const float* sink, int HB, int LD, int split, float* part) {
  static size_t reserved = 0;
  if (smem > 48 * 1024 && smem > reserved) {
    if (hipFuncSetAttribute((const void*)latent_attention_mfma_kernel<RT, DKS, WHOLE>, hipFuncAttributeMaxDynamicSharedMemorySize,
                            (int)smem) != hipSuccess)
      JLLM_FAIL("latent_attention: cannot reserve %zu bytes of LDS", smem);
    reserved = smem;
  }
  latent_attention_mfma_kernel<RT, DKS, WHOLE><<<grid, LM_WAVES * 64, smem, stream>>>(
      (const bf16_t*)qa, ldq, (bf16_t*)out, ldo, (const bf16_t*)cache, block_table, max_blocks, tiles, positions, H, R, Dk,
      page_size, window, scale, sink, HB, LD, split, part);
  return 0;
}

template <int RT, int DKS>
static int lm_launch(dim3 grid, size_t smem, hipStream_t stream, const void* qa, int ldq, void* out, int ldo, const void* cache,
                     const int* block_table, int max_blocks, const int* tiles, const int* positions, int H, int R, int Dk,
                     int page_size, int window, float scale, const float* sink, int HB, int LD, int split, float* part) {
  return R == RT * 16 && Dk == DKS * 32
             ? lm_launch_as<RT, DKS, true>(grid, smem, stream, qa, ldq, out, ldo, cache, block_table, max_blocks, tiles, positions, H, R, Dk, page_size, window, scale, sink, HB, LD, split, part)
             : lm_launch_as<RT, DKS, false>(grid, smem, stream, qa, ldq, out, ldo, cache, block_table, max_blocks, tiles, positions, H, R, Dk, page_size, window, scale, sink, HB, LD, split, part);
}

template <int NJ, int DKS>
static int lm_launch_rows(dim3 grid, hipStream_t stream, const void* qa, int ldq, void* out, int ldo, const void* cache,
                          const int* block_table, int max_blocks, const int* tiles, const int* positions, int H, int R, int Dk,
                          int page_size, int window, float scale, const float* sink, int HB, int n_hb) {
  static size_t reserved = 0;
  const size_t smem = ((size_t)2 * LM_KEYS * (DKS * 32 + 16) + 64 * LM_PS) * sizeof(bf16_t) + 768 * sizeof(float);
  if (smem > 48 * 1024 && smem > reserved) {
    if (hipFuncSetAttribute((const void*)latent_attention_rows_kernel<NJ, DKS>, hipFuncAttributeMaxDynamicSharedMemorySize,
                            (int)smem) != hipSuccess)
      JLLM_FAIL("latent_attention: cannot reserve %zu bytes of LDS", smem);
    reserved = smem;
  }
  latent_attention_rows_kernel<NJ, DKS><<<grid, LM_WAVES * 64, smem, stream>>>(
      (const bf16_t*)qa, ldq, (bf16_t*)out, ldo, (const bf16_t*)cache, block_table, max_blocks, tiles, positions, H, R, Dk,
      page_size, window, scale, sink, HB, n_hb);
  return 0;
}

// returns 0 when it ran, 1 when the shape is not one it takes (the caller uses the general kernel), -1 on errors
extern "C" int jllm_latent_attention_bf16(const void* qa, int ldq, void* out, int ldo, const void* cache,
                                          const int* block_table, int max_blocks, const int* tiles, const int* positions,
                                          int n_tiles, int tile_rows, int H, int R, int Dk, int page_size, int window,
                                          float scale, const float* sink, int split, int n_z, float* part,
                                          hipStream_t stream) {
  if (n_tiles <= 0) return 0;
  if (tile_rows != LM_TILE_ROWS) JLLM_FAIL("latent_attention: runs of %d rows, this kernel takes %d", tile_rows, LM_TILE_ROWS);
  if (H <= 0 || R <= 0 || Dk < R || window < 0 || page_size <= 0 || max_blocks <= 0) JLLM_FAIL("latent_attention: H %d R %d Dk %d window %d", H, R, Dk, window);
  if ((R & 15) || (Dk & 7) || R > 512 || Dk > 576 || (page_size & (page_size - 1))) return 1;  // (longer rows: two blocks of keys exceed the LDS)
  if (((uintptr_t)qa & 15) || ((uintptr_t)cache & 15) || ((uintptr_t)out & 7) || (ldq & 7) || (ldo & 3)) return 1;
  if (ldq < H * Dk || ldo < H * R) JLLM_FAIL("latent_attention: row strides %d/%d", ldq, ldo);
  int HB = 1;
  while (HB < H && HB < 64) HB <<= 1;
  const int RW = 64 / HB;
  const int n_hb = (H + HB - 1) / HB, n_rg = (LM_TILE_ROWS + RW - 1) / RW;
  if ((long)n_hb * n_rg > 65535) return 1;
  // staged rows lie (Dk rounded up to 32) + pad elements apart, with the stride = 16 mod 64 elements (8 mod 32 words):
  // four consecutive rows of a transposing load then cover all banks
  const int dkp = (Dk + 31) & ~31;
  int LD = dkp + 16;
  while ((LD & 63) != 16) LD += 8;
  const size_t smem = (size_t)2 * LM_KEYS * LD * sizeof(bf16_t);  // two buffers that take turns
  // `split` < 0: runs of up to tile_rows rows. Otherwise every tile is a single row (the caller's promise); > 0: whose keys are cut into absolute ranges of `split`
  // keys over n_z workgroups; `part` holds rows x H x n_z x (R + 4) floats
  if (split > 0 && ((split & 63) || n_z < 1 || n_z > 64 || !part)) JLLM_FAIL("latent_attention: ranges of %d keys over %d workgroups", split, n_z);
  dim3 grid(n_tiles, n_hb * (split < 0 ? n_rg : 1), split > 0 ? n_z : 1);
  int rc;
  if (split < 0)
    // The smallest instance that holds the sizes; what it pads is multiplied as zeros. 2,048 rows, against the kernel for
    // single rows, which took these runs too: 4 heads of 64 + 32 entries 90 -> 60 us (padded to 256 entries 67), 8 of 128 + 64
    // 123 -> 70, 3 of 144 + 24 (padded to 512 + 64) 173 -> 101, 16 of 256 + 64 364 -> 189. What that kernel did faster are rows
    // alone and a few rows of a new prompt where latents are short and heads few: 30 rows and three single rows of 1,500 keys with
    // 4 heads of 64 + 32 30 -> 44, 3 of 144 + 24 61 -> 70, 8 of 256 + 64 69 -> 71, 16 of 512 + 64 85 -> 73; 20 rows 5.0 -> 6.1,
    // 7.8 -> 8.7, 9.9 -> 10.3, 15.6 -> 13.8.
    rc = R <= 128 && dkp <= 128
             ? lm_launch_rows<1, 4>(grid, stream, qa, ldq, out, ldo, cache, block_table, max_blocks, tiles, positions, H, R, Dk, page_size, window, scale, sink, HB, n_hb)
         : R <= 128 && dkp <= 256
             ? lm_launch_rows<1, 8>(grid, stream, qa, ldq, out, ldo, cache, block_table, max_blocks, tiles, positions, H, R, Dk, page_size, window, scale, sink, HB, n_hb)
             : lm_launch_rows<4, 18>(grid, stream, qa, ldq, out, ldo, cache, block_table, max_blocks, tiles, positions, H, R, Dk, page_size, window, scale, sink, HB, n_hb);
  else if (R <= 64 && dkp <= 128)
    rc = lm_launch<4, 4>(grid, smem, stream, qa, ldq, out, ldo, cache, block_table, max_blocks, tiles, positions, H, R, Dk, page_size, window, scale, sink, HB, LD, split, part);
  else if (R <= 128 && dkp <= 256)
    rc = lm_launch<8, 8>(grid, smem, stream, qa, ldq, out, ldo, cache, block_table, max_blocks, tiles, positions, H, R, Dk, page_size, window, scale, sink, HB, LD, split, part);
  else
    rc = lm_launch<32, 18>(grid, smem, stream, qa, ldq, out, ldo, cache, block_table, max_blocks, tiles, positions, H, R, Dk, page_size, window, scale, sink, HB, LD, split, part);
  if (rc != 0) return rc;
  JLLM_CHECK_LAUNCH("latent_attention");
  if (split > 0) {
    latent_attention_merge_kernel<<<dim3(n_tiles, H), 256, 0, stream>>>(part, positions, H, R, window, split, n_z, sink, (bf16_t*)out, ldo);
    JLLM_CHECK_LAUNCH("latent_attention_merge");
  }
  return 0;
}
