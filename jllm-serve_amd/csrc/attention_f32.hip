// Causal grouped-query attention over a paged cache, fp32, head size 128: the two kernels that the 32-bit path takes at
// the head size of its models. A row's result has the same bits from either of them and from the general kernel
// (attention_generic.hip), whatever the step's other rows are: the walk over the keys (64-key blocks aligned to absolute
// positions, wave w of four takes the blocks c with c % 4 == w), the order of every sum (dot products in ascending dims, the
// block's probabilities over a tree of lanes 32, 16, .. 1 apart, weighted sums in ascending keys, the waves' results
// in the order of the waves) and what is one multiply-add are the general kernel's. Cache layout and table as there.
//
//  * single rows (decode steps): a workgroup per row and up to four heads of a kv head, a lane per key. The general kernel
//    waits for a handful of 16-byte loads at a time; here a lane requests its whole key row at once, or has it by way of LDS, and a
//    block's values in four groups of 16 keys, each on its way while the one before is used. Three rows of 90, 246 and 400 keys, 16
//    heads over 8, inside a graph: the general kernel (with a score bias of zeros, which it alone takes) 39.4 us, here 11.5; of 400
//    keys each 39.5 / 11.6.
//  * many rows (portions): a workgroup takes 16 query vectors (rows of one request x the heads of a kv head), so a key is
//    read once for all of them instead of once per row, and both products run on the matrix cores' fp32 form, whose sums
//    are chains of multiply-adds in ascending order (see gemm_generic.hip). Three prompts of 847 rows in all, 16 heads over 8:
//    188 -> 54 us; the multiplies alone take a third of that, the rest is keys and values on their way from the L2.
#include <math.h>

#include "common.h"
#include "lds_ring.h"

#define AF_HD 128
#define AF_WAVES 4

typedef float floatx4 __attribute__((ext_vector_type(4)));

struct AttF32 {
  const float* q;
  float* out;
  const float *k, *v;
  const int *table, *row_req, *positions;
  int ldq, ldo, max_blocks, n_tokens, H, Hkv, page_size, window;
  float scale;
};

// where position j of the request with this table row lies, in rows of AF_HD
__device__ __forceinline__ int cache_row(const AttF32& A, const int* __restrict__ tbl, int kvh, int j) {
  return (tbl[j / A.page_size] * A.Hkv + kvh) * A.page_size + j % A.page_size;
}

// ---------------------------------------------------------------------------------------------- single rows

// STAGED: the keys come by way of LDS. A lane that reads a key's row takes 16 bytes of a line at a time, 64 lines at once: the
// four waves' 128 KB do not stay in the first-level cache (32 KB) until a line's other pieces are asked for, so each crosses from
// the L2 several times. In LDS they come once, in whole lines, and the next block's while this one's values are weighted; but a
// compute unit then holds one workgroup. Registers / LDS, 16 heads over 8: 300 keys 12.1 / 11.2 us, three rows of 400 14.2 /
// 11.8, of 2,000 56.1 / 41.1, 16 of 1,000 30.6 / 25.6; where there are more workgroups than compute units, 64 of 1,000 93.2 / 94.8
// and 64 of 100 12.1 / 17.7.
// `key_rows`, where STAGED: [AF_WAVES][64 keys][512 bytes]; `mg`: every wave's maximum, sum and weighted sums.
template <int GC, bool STAGED>
__device__ __forceinline__ void attention_rows(const AttF32& A, unsigned char* key_rows, float (&qs)[GC][AF_HD], float (&mg)[AF_WAVES][GC][2 + AF_HD]) {
  const int t = blockIdx.x, lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int G = A.H / A.Hkv, chunks = (G + GC - 1) / GC;
  const int kvh = blockIdx.y / chunks;
  const int h0 = kvh * G + (blockIdx.y % chunks) * GC;
  const int gn = min(GC, kvh * G + G - h0);  // a spare place does the last head again and is not stored
  const int pos = A.positions[t];
  const int* tbl = A.table + (size_t)A.row_req[t] * A.max_blocks;
  const int first = A.window > 0 ? max(0, pos + 1 - A.window) : 0;
  const int b_first = first >> 6;
  int blk = b_first + ((wave - b_first) & (AF_WAVES - 1));
  // every lane names a key inside the row's range: those beyond it repeat the nearest one with probability 0
  auto row_of = [&](int b) { return cache_row(A, tbl, kvh, min(max(b * 64 + lane, first), pos)); };
  int row = row_of(blk);
  for (int i = threadIdx.x; i < GC * AF_HD; i += 64 * AF_WAVES)
    qs[i / AF_HD][i % AF_HD] = A.q[(size_t)t * A.ldq + (size_t)(h0 + min(i / AF_HD, gn - 1)) * AF_HD + i % AF_HD];
  __syncthreads();
  float acc[GC][2], m[GC], l[GC];
#pragma unroll
  for (int g = 0; g < GC; ++g) m[g] = -INFINITY, l[g] = 0.f, acc[g][0] = acc[g][1] = 0.f;
  // A block's keys go into the wave's own 32 KB of LDS, two rows (1 KB) a load, piece j (16 bytes) of key k at place j ^ (k % 32):
  // read back a lane per key, a row apart, neighbouring lanes meet different banks.
  unsigned char* keys = key_rows + wave * 64 * AF_HD * 4;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const unsigned char*)keys;
  auto request_keys = [&](int row) {
#pragma unroll
    for (int c = 0; c < 32; ++c) {
      const int r0 = __builtin_amdgcn_readlane(row, 2 * c), r1 = __builtin_amdgcn_readlane(row, 2 * c + 1);
      const int piece = (lane & 31) ^ ((2 * c + (lane >> 5)) & 31);
      const float* src = A.k + (size_t)(lane < 32 ? r0 : r1) * AF_HD + piece * 4;
      load_to_lds_16(src, lds0 + c * 1024u);
    }
  };
  if (STAGED && blk * 64 <= pos) request_keys(row);
  for (; blk * 64 <= pos; blk += AF_WAVES) {
    const int c0 = blk * 64, kj = c0 + lane;
    const bool valid = kj >= first && kj <= pos;
    const int next = blk + AF_WAVES;
    auto fetch = [&](float (&vv)[16][2], int jb) {
#pragma unroll
      for (int u = 0; u < 16; ++u) {
        const float* vr = A.v + (size_t)__builtin_amdgcn_readlane(row, jb + u) * AF_HD;
        vv[u][0] = vr[lane];
        vv[u][1] = vr[lane + 64];
      }
    };
    const floatx4* kr = (const floatx4*)(A.k + (size_t)row * AF_HD);
    floatx4 kv[STAGED ? 1 : AF_HD / 4];
    float va[16][2], vb[16][2];
    int next_row = row;
    if constexpr (STAGED) {
      wait_loads<0>();  // the block's keys
      __builtin_amdgcn_sched_barrier(0);
      fetch(va, 0);
      next_row = row_of(next);
    } else {
#pragma unroll
      for (int i = 0; i < AF_HD / 4; ++i) kv[i] = kr[i];
    }
    __builtin_amdgcn_sched_barrier(0);
    float d[GC], p[GC];
#pragma unroll
    for (int g = 0; g < GC; ++g) d[g] = 0.f;
    constexpr int AT_ONCE = STAGED ? 8 : 4;  // pieces at a time: all of the queries' (and the keys') LDS reads would take all registers
#pragma unroll
    for (int i0 = 0; i0 < AF_HD / 4; i0 += AT_ONCE) {
      floatx4 part[AT_ONCE];
#pragma unroll
      for (int i = 0; i < AT_ONCE; ++i) {
        if constexpr (STAGED)
          part[i] = *(const floatx4*)(keys + lane * AF_HD * 4 + (((i0 + i) ^ (lane & 31)) << 4));
        else
          part[i] = kv[i0 + i];
      }
#pragma unroll
      for (int i = 0; i < AT_ONCE; ++i)
#pragma unroll
        for (int g = 0; g < GC; ++g) {
          const floatx4 qv = *(const floatx4*)&qs[g][4 * (i0 + i)];
#pragma unroll
          for (int e = 0; e < 4; ++e) d[g] = fmaf(qv[e], part[i][e], d[g]);
        }
#pragma unroll
      for (int g = 0; g < GC; ++g) asm volatile("" : "+v"(d[g]));  // (nor does the chain sink below to where its sum is used)
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (!STAGED) {
      fetch(va, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int g = 0; g < GC; ++g) {
#pragma clang fp contract(off)
      const float s = valid ? d[g] * A.scale : -INFINITY;
      const float m_new = fmaxf(m[g], wave_max(s));
      p[g] = valid ? expf(s - m_new) : 0.f;
      const float alpha = expf(m[g] - m_new);
      l[g] = fmaf(l[g], alpha, wave_sum(p[g]));
      acc[g][0] *= alpha;
      acc[g][1] *= alpha;
      m[g] = m_new;
    }
    const int j0 = max(0, first - c0), j1 = min(63, pos - c0);
    auto use = [&](const float (&vv)[16][2], int jb) {
#pragma unroll
      for (int u4 = 0; u4 < 16; u4 += 4) {
        if (jb + u4 + 3 < j0 || jb + u4 > j1) continue;  // (in fours, as the general kernel: p = 0 of a key outside is multiplied)
#pragma unroll
        for (int u = u4; u < u4 + 4; ++u)
#pragma unroll
          for (int g = 0; g < GC; ++g) {
            const float pj = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(p[g]), jb + u));
            acc[g][0] = fmaf(pj, vv[u][0], acc[g][0]);
            acc[g][1] = fmaf(pj, vv[u][1], acc[g][1]);
          }
      }
    };
    fetch(vb, 16);
    __builtin_amdgcn_sched_barrier(0);
    use(va, 0);
    fetch(va, 32);
    __builtin_amdgcn_sched_barrier(0);
    use(vb, 16);
    fetch(vb, 48);
    if constexpr (STAGED) {
      // The next keys go out with nothing else on its way: the compiler does not count loads into LDS, and would wait for these
      // where it waits for values. Every read of the last keys is done, their products are.
      __builtin_amdgcn_sched_barrier(0);
      row = next_row;
      __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
      if (next * 64 <= pos) request_keys(row);
    } else {
      if (next * 64 <= pos) row = row_of(next);
    }
    __builtin_amdgcn_sched_barrier(0);
    use(va, 32);
    use(vb, 48);
  }
#pragma unroll
  for (int g = 0; g < GC; ++g) {
    if (lane == 0) mg[wave][g][0] = m[g], mg[wave][g][1] = l[g];
    mg[wave][g][2 + lane] = acc[g][0];
    mg[wave][g][2 + lane + 64] = acc[g][1];
  }
  __syncthreads();
  for (int i = threadIdx.x; i < gn * AF_HD; i += 64 * AF_WAVES) {
    const int g = i / AF_HD, dim = i % AF_HD;
    float mm = mg[0][g][0], ll = mg[0][g][1], x = mg[0][g][2 + dim];
#pragma unroll
    for (int w = 1; w < AF_WAVES; ++w) {
#pragma clang fp contract(off)
      const float om = mg[w][g][0], ol = mg[w][g][1];
      if (ol == 0.f) continue;  // that wave had no key
      const float m_new = fmaxf(mm, om);
      const float ca = expf(mm - m_new), cb = expf(om - m_new);
      ll = fmaf(ll, ca, ol * cb);
      x = fmaf(x, ca, mg[w][g][2 + dim] * cb);
      mm = m_new;
    }
    A.out[(size_t)t * A.ldo + (size_t)(h0 + g) * AF_HD + dim] = x * (1.0f / ll);
  }
}

// STAGED: rows of more than two blocks of keys by way of LDS. The host knows the table's width alone, and a captured step's is that
// of its bucket, however short the rows are: the row itself decides. Registers / LDS in that kernel, a row of 16 heads over 8: 20 keys
// 4.9 / 6.0 us, 60 keys 5.6 / 6.3, 120 keys 6.6 / 6.6, 200 keys 8.3 / 7.3, 256 keys 8.9 / 7.3; 16 rows of 60 5.7 / 6.5, of 250 9.7 / 8.4.
template <int GC, bool STAGED>
__global__ __launch_bounds__(64 * AF_WAVES, STAGED ? 1 : 2) void attention_f32_rows_kernel(AttF32 A) {
  extern __shared__ __align__(1024) unsigned char key_rows[];
  __shared__ __align__(16) float qs[GC][AF_HD];
  __shared__ float mg[AF_WAVES][GC][2 + AF_HD];
  if constexpr (STAGED) {
    const int pos = A.positions[blockIdx.x];
    const int first = A.window > 0 ? max(0, pos + 1 - A.window) : 0;
    if ((pos >> 6) - (first >> 6) >= 2) {
      attention_rows<GC, true>(A, key_rows, qs, mg);
      return;
    }
  }
  attention_rows<GC, false>(A, nullptr, qs, mg);
}

// ---------------------------------------------------------------------------------------------- many rows

// lane group q (of 16 lanes) holds x[j] = X[q][j]; afterwards x[s] = X[s][q]. v_permlane32_swap exchanges the upper half of
// its first register with the lower half of its second, v_permlane16_swap the odd groups with the even ones.
__device__ __forceinline__ floatx4 lanes_transposed(floatx4 x) {
  auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(x[0]), __float_as_uint(x[2]), false, false);
  auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(x[1]), __float_as_uint(x[3]), false, false);
  auto lo = __builtin_amdgcn_permlane16_swap(a[0], b[0], false, false);
  auto hi = __builtin_amdgcn_permlane16_swap(a[1], b[1], false, false);
  return floatx4{__uint_as_float(lo[0]), __uint_as_float(lo[1]), __uint_as_float(hi[0]), __uint_as_float(hi[1])};
}

__device__ __forceinline__ floatx4 mfma_f32(float a, float b, floatx4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

// Column c of a wave's products is query vector c: row c / G of the tile, head c % G of the kv head; lane l holds column
// l % 16. Scores: D[key][c] += K[key][dims] q[c][dims], four tiles of 16 keys, 32 steps of four dims each; lane l then has
// keys 16 t + 4 (l / 16) + i. Weighted sums: D[dim][c] += V^T[dim][key] p[c][key]; a lane's 16 bytes of V are four
// neighbouring dims of one key, which go to four tiles (a tile's row r is dim 4 r + j of its 64 dims), so V needs no
// transposition; keys and probabilities are transposed over the lane groups in registers.
//
// A workgroup takes the rows that a tile begins with, as many as are one request's. What else lies in the tile is the work of
// the first `spread` workgroups (SPREAD: where there are several requests), one for each request: it looks for the places
// inside tiles where its request's rows begin. A workgroup that walked all of its tile's requests in turn made the step
// wait for it: 20 rows of a prompt and five single rows of up to 400 keys 71 us, here 24 (the general kernel: 41); 32 single rows of
// 1,000 to 2,860 keys behind 2,000 rows of a prompt 1,050, here 355 (1,770); 64 requests of 32 rows, where there is nothing
// to find, 52, here 58 (195), eight of 32 rows behind 500 keys 37, here 47 (152): the workgroups that find nothing stand in front
// of tiles. (All of them in front of all tiles, or behind them where all are resident: these two 129 instead of 134 and 37, but
// single rows behind portions 2 to 6 % slower.)
template <bool SPREAD>
__global__ __launch_bounds__(64 * AF_WAVES, 2) void attention_f32_tiles_kernel(AttF32 A, int rows, int spread) {
  __shared__ __align__(16) float mg[AF_WAVES][16][4 + AF_HD];  // every wave's maximum, sum (and two spare places), weighted sums
  __shared__ int found[AF_WAVES];
  const int lane = threadIdx.x & 63, col = lane & 15, quad = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int G = A.H / A.Hkv, kvh = blockIdx.y;
  const bool inner = SPREAD && (int)blockIdx.x < spread;
  int t0 = inner ? 0 : ((int)blockIdx.x - (SPREAD ? spread : 0)) * rows;
  for (;; ++t0) {
    if (__builtin_expect(inner, 0)) {  // the next row inside a tile with which rows of this request begin
      int at = 0x7fffffff;
      for (; t0 < A.n_tokens; t0 += 8 * 64 * AF_WAVES) {
        int before[8], here[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          const int t = min(t0 + u * 64 * AF_WAVES + (int)threadIdx.x, A.n_tokens - 1);
          before[u] = A.row_req[max(t - 1, 0)], here[u] = A.row_req[t];
        }
#pragma unroll
        for (int u = 7; u >= 0; --u) {
          const int t = t0 + u * 64 * AF_WAVES + (int)threadIdx.x;
          if (t < A.n_tokens && here[u] == (int)blockIdx.x && before[u] != here[u] && t % rows != 0) at = t;
        }
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) at = min(at, __shfl_xor(at, o, 64));
        if (lane == 0) found[wave] = at;
        __syncthreads();
#pragma unroll
        for (int w = 0; w < AF_WAVES; ++w) at = min(at, found[w]);
        at = __builtin_amdgcn_readfirstlane(at);
        __syncthreads();
        if (at != 0x7fffffff) break;
      }
      if (at == 0x7fffffff) return;
      t0 = at;
    }
    const int end = min(inner ? rows - t0 % rows : rows, A.n_tokens - t0);  // rows of the tile from here on
    const int ri = min(col / G, end - 1);  // this lane's row of those taken ...
    const int head = kvh * G + col % G;     // ... and head
    floatx4 qf[AF_HD / 16];                // the lane's query vector at dims 16 c + 4 s + quad
    {
      const floatx4* qr = (const floatx4*)(A.q + (size_t)(t0 + ri) * A.ldq + (size_t)head * AF_HD);
#pragma unroll
      for (int c = 0; c < AF_HD / 16; ++c) qf[c] = qr[4 * c + quad];
    }
    // lane i of every 16 looks at row i: how many belong to the first one's request, and which keys they see
    const int ti = t0 + min(col, end - 1), req_i = A.row_req[ti], pos_i = A.positions[ti];
    const int req = __builtin_amdgcn_readfirstlane(req_i);
    const int n = min(end, __builtin_ctz(~((uint32_t)__ballot(req_i == req) & 0xffffu)));
    const int first_i = A.window > 0 ? max(0, pos_i + 1 - A.window) : 0;
    int low = col < n ? first_i : 0x7fffffff, low_pos = col < n ? pos_i : 0x7fffffff;
    int high = col < n ? pos_i : -1, last_first = col < n ? first_i : 0;
#pragma unroll
    for (int o = 8; o > 0; o >>= 1) {
      low = min(low, __shfl_xor(low, o, 64)), low_pos = min(low_pos, __shfl_xor(low_pos, o, 64));
      high = max(high, __shfl_xor(high, o, 64)), last_first = max(last_first, __shfl_xor(last_first, o, 64));
    }
    low = __builtin_amdgcn_readfirstlane(low), low_pos = __builtin_amdgcn_readfirstlane(low_pos);
    high = __builtin_amdgcn_readfirstlane(high), last_first = __builtin_amdgcn_readfirstlane(last_first);
#pragma unroll
    for (int c = 0; c < AF_HD / 16; ++c) qf[c] = lanes_transposed(qf[c]);
    const int* tbl = A.table + (size_t)req * A.max_blocks;
    const bool mine = col / G < n;
    const int pos = mine ? A.positions[t0 + ri] : -1;  // a lane without a row sees no key
    const int first = mine && A.window > 0 ? max(0, pos + 1 - A.window) : 0;
    floatx4 acc[2][4];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[h][j] = floatx4{0.f, 0.f, 0.f, 0.f};
    float m = -INFINITY, l = 0.f;
    const int b_first = low >> 6;
    for (int blk = b_first + ((wave - b_first) & (AF_WAVES - 1)); blk * 64 <= high; blk += AF_WAVES) {
      const int c0 = blk * 64;
      const int row = cache_row(A, tbl, kvh, min(max(c0 + lane, low), high));  // key c0 + lane, or the nearest that some row sees
      floatx4 s[4];
      floatx4 kf[4][AF_HD / 16];
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const floatx4* kr = (const floatx4*)(A.k + (size_t)__shfl(row, 16 * t + col, 64) * AF_HD);
#pragma unroll
        for (int c = 0; c < AF_HD / 16; ++c) kf[t][c] = kr[4 * c + quad];
        s[t] = floatx4{0.f, 0.f, 0.f, 0.f};
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int t = 0; t < 4; t += 2) {
#pragma unroll
        for (int c = 0; c < AF_HD / 16; ++c) {
          const floatx4 ka = lanes_transposed(kf[t][c]), kb = lanes_transposed(kf[t + 1][c]);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            s[t] = mfma_f32(ka[e], qf[c][e], s[t]);
            s[t + 1] = mfma_f32(kb[e], qf[c][e], s[t + 1]);
          }
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      // values of 16 keys (t): lane's key 16 t + 4 u + quad, dims 64 h + 4 col .. + 3
      auto fetch = [&](floatx4 (&vv)[4][2], int t) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const float* vr = A.v + (size_t)__shfl(row, 16 * t + 4 * u + quad, 64) * AF_HD + 4 * col;
          vv[u][0] = *(const floatx4*)vr;
          vv[u][1] = *(const floatx4*)(vr + 64);
        }
      };
      floatx4 va[4][2], vb[4][2];
      fetch(va, 0);
      fetch(vb, 1);
      __builtin_amdgcn_sched_barrier(0);
      const bool any = c0 <= pos && c0 + 63 >= first;  // this lane's row sees a key of the block
      float m_new, alpha;
      {
#pragma clang fp contract(off)
        float top = -INFINITY;
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int key = c0 + 16 * t + 4 * quad + i;
            s[t][i] = key >= first && key <= pos ? s[t][i] * A.scale : -INFINITY;
            top = fmaxf(top, s[t][i]);
          }
        top = fmaxf(top, __shfl_xor(top, 16, 64));
        top = fmaxf(top, __shfl_xor(top, 32, 64));
        m_new = any ? fmaxf(m, top) : m;
        alpha = any ? expf(m - m_new) : 1.f;
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
          for (int i = 0; i < 4; ++i) s[t][i] = s[t][i] == -INFINITY ? 0.f : expf(s[t][i] - m_new);
        // the sum over the block's 64 keys, key k with k ^ 32 first, then k ^ 16, .. k ^ 1
        float x[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          x[i] = (s[0][i] + s[2][i]) + (s[1][i] + s[3][i]);
          x[i] += __shfl_xor(x[i], 32, 64);
          x[i] += __shfl_xor(x[i], 16, 64);
        }
        l = fmaf(l, alpha, (x[0] + x[2]) + (x[1] + x[3]));
        m = m_new;
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[h][j][i] *= alpha;
      }
      // a key that some of the rows do not see is multiplied by 0 for them, which an infinite value would not survive
      const bool partial = c0 < last_first || c0 + 63 > low_pos;
      auto use = [&](const floatx4 (&vv)[4][2], int t) {
        const floatx4 pt = lanes_transposed(s[t]);  // pt[u]: key 16 t + 4 u + quad
        if (partial) {
          bool odd = false;
#pragma unroll
          for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
              for (int j = 0; j < 4; ++j) odd = odd || !(fabsf(vv[u][h][j]) < INFINITY);
          if (__ballot(odd)) {  // (rare) key by key, for the rows that see it
#pragma unroll 1
            for (int k = 0; k < 16; ++k) {
              const int key = c0 + 16 * t + k;
              const float pk = k < 8 ? (k < 4 ? pt[0] : pt[1]) : (k < 12 ? pt[2] : pt[3]);
              const float pe = __shfl(pk, col + 16 * (k & 3), 64);
              const float* vr = A.v + (size_t)__shfl(row, 16 * t + k, 64) * AF_HD;
#pragma unroll
              for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int j = 0; j < 4; ++j)
#pragma unroll
                  for (int i = 0; i < 4; ++i)
                    if (key >= first && key <= pos) acc[h][j][i] = fmaf(pe, vr[64 * h + 4 * (4 * quad + i) + j], acc[h][j][i]);
            }
            return;
          }
        }
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
          for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int j = 0; j < 4; ++j) acc[h][j] = mfma_f32(vv[u][h][j], pt[u], acc[h][j]);
      };
      use(va, 0);
      fetch(va, 2);
      __builtin_amdgcn_sched_barrier(0);
      use(vb, 1);
      fetch(vb, 3);
      __builtin_amdgcn_sched_barrier(0);
      use(va, 2);
      use(vb, 3);
    }
    if (quad == 0) mg[wave][col][0] = m, mg[wave][col][1] = l;
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int i = 0; i < 4; ++i)  // dims 64 h + 4 (4 quad + i) .. + 3 lie in the four tiles
        *(floatx4*)&mg[wave][col][4 + 64 * h + 16 * quad + 4 * i] = floatx4{acc[h][0][i], acc[h][1][i], acc[h][2][i], acc[h][3][i]};
    __syncthreads();
    {
      const int c = threadIdx.x >> 4, r = c / G, d0 = (threadIdx.x & 15) * 8;
      if (r < n) {
        float mm = mg[0][c][0], ll = mg[0][c][1], x[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) x[i] = mg[0][c][4 + d0 + i];
#pragma unroll
        for (int w = 1; w < AF_WAVES; ++w) {
#pragma clang fp contract(off)
          const float om = mg[w][c][0], ol = mg[w][c][1];
          if (ol == 0.f) continue;
          const float m_new = fmaxf(mm, om);
          const float ca = expf(mm - m_new), cb = expf(om - m_new);
          ll = fmaf(ll, ca, ol * cb);
#pragma unroll
          for (int i = 0; i < 8; ++i) x[i] = fmaf(x[i], ca, mg[w][c][4 + d0 + i] * cb);
          mm = m_new;
        }
        const float inv = 1.0f / ll;
        float* o = A.out + (size_t)(t0 + r) * A.ldo + (size_t)(kvh * G + c % G) * AF_HD + d0;
#pragma unroll
        for (int i = 0; i < 8; ++i) o[i] = x[i] * inv;
      }
    }
    if (!inner) return;
    __syncthreads();
  }
}

template <int GC, bool STAGED>
static int launch_rows(const AttF32& A, dim3 grid, hipStream_t stream) {
  constexpr int smem = STAGED ? AF_WAVES * 64 * AF_HD * 4 : 0;
  if constexpr (STAGED) {
    static bool configured = false;
    if (!configured) {  // above 64 KB the size has to be allowed first
      if (hipFuncSetAttribute((const void*)attention_f32_rows_kernel<GC, true>, hipFuncAttributeMaxDynamicSharedMemorySize, smem) != hipSuccess)
        JLLM_FAIL("attention_f32: cannot reserve %d bytes of LDS", smem);
      configured = true;
    }
  }
  attention_f32_rows_kernel<GC, STAGED><<<grid, 64 * AF_WAVES, smem, stream>>>(A);
  JLLM_CHECK_LAUNCH("attention_f32");
  return 0;
}

// fp32, head size 128, 16-byte aligned rows; returns 1 for what it leaves to the general kernel. `n_requests` bounds
// row_req, the block table's width the keys. Which kernel: a tile holds 16 / G rows of one request, and reads their keys
// once; where the rows are spread over as many requests (steps of single tokens) there is nothing to share and a workgroup
// per row has more waves. A portion of few rows goes row by row too: a tile's chain is about 12 us for the first 64 keys, a
// row's 5.5, as long as its workgroups (row x head) are one per compute unit, a few where the keys are few. 16 heads over
// 8, rows / tiles (the general kernel): 4 rows of a new prompt 5.5 / 11.7 us (6.8), 20 rows 5.9 / 12.1 (10.2), 64 rows 8.4 /
// 12.3, 96 rows 16.0 / 13.1; 20 rows behind 200 keys 13.2 / 15.1, 40 rows 17.6 / 15.3; 16 rows behind 1,000 keys 31.6 (25.6 by way of LDS) / 39.6,
// 20 rows 46.7 / 41.6. Up to 16 keys the general kernel lies between: 64 rows of eight new prompts, 24 heads over 3, 9.8 us,
// 11.8 by rows, 12.5 by tiles.
extern "C" int jllm_attention_f32(const void* q, int ldq, void* out, int ldo, const void* kcache, const void* vcache, const int* block_table,
                                  int max_blocks, const int* row_req, const int* positions, int n_tokens, int n_requests, int H,
                                  int Hkv, int hd, int page_size, int window, float scale, hipStream_t stream) {
  if (n_tokens <= 0) return 0;
  if (hd != AF_HD || H <= 0 || Hkv <= 0 || H % Hkv != 0 || page_size <= 0 || max_blocks <= 0 || window < 0 || n_requests <= 0) return 1;
  if (ldq < H * hd || ldo < H * hd || (ldq & 3) || H > 65535) return 1;
  if (((uintptr_t)q | (uintptr_t)kcache | (uintptr_t)vcache) & 15) return 1;
  const AttF32 A = {(const float*)q, (float*)out, (const float*)kcache, (const float*)vcache, block_table, row_req, positions,
                    ldq, ldo, max_blocks, n_tokens, H, Hkv, page_size, window, scale};
  const int G = H / Hkv;
  int cus = jllm_compute_units();
  if (cus <= 0) cus = 256;
  const long keys = (long)max_blocks * page_size;  // no row sees more
  const long pairs = (long)n_tokens * H;
  const bool few = pairs <= (long)cus * (keys <= 64 ? 5 : keys <= 256 ? 2 : 1);
  if (G <= 8 && n_tokens >= 4 * n_requests && !few) {
    if (keys <= 16 && pairs <= 6L * cus) return 1;
    const int rows = 16 / G;
    const int tiles = (n_tokens + rows - 1) / rows;
    if (n_requests > 1)
      attention_f32_tiles_kernel<true><<<dim3(tiles + n_requests, Hkv), 64 * AF_WAVES, 0, stream>>>(A, rows, n_requests);
    else
      attention_f32_tiles_kernel<false><<<dim3(tiles, Hkv), 64 * AF_WAVES, 0, stream>>>(A, rows, 0);
  } else if (pairs <= cus && keys > 256) {  // one round of workgroups, more than a block a wave
    return launch_rows<1, true>(A, dim3(n_tokens, H), stream);
  } else {  // heads share a workgroup where the step still has two workgroups for every compute unit, as in the general kernel
    if (G >= 3 && (long)n_tokens * Hkv * ((G + 3) / 4) >= 2L * cus)
      return launch_rows<4, false>(A, dim3(n_tokens, Hkv * ((G + 3) / 4)), stream);
    else if (G >= 2 && (G <= 4 || keys > 64) && (long)n_tokens * Hkv * ((G + 1) / 2) >= 2L * cus)
      return launch_rows<2, false>(A, dim3(n_tokens, Hkv * ((G + 1) / 2)), stream);
    else
      return launch_rows<1, false>(A, dim3(n_tokens, H), stream);
  }
  JLLM_CHECK_LAUNCH("attention_f32");
  return 0;
}
