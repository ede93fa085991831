// The attention of attention_dv.hip for steps of single rows (decode) at key size 128 and value size 128 or 256, bf16 cache,
// on the matrix cores: what attention_dv_mfma.hip does there, without its tile of 32 rows of which one is there.
//
// A workgroup takes a row, a key slot and a share of the row's 64-key blocks (numbered as there: the blocks of kept first
// keys, then the window's); the query heads that read the key slot, up to 16, are the columns of the products. Per block a
// wave takes 16 keys: S^T[key][head] = K Q^T is four v_mfma_f32_16x16x32_bf16 with K straight from the cache as the A operand
// (lane l: key l % 16, dims 32 j + (l / 16) 8 .. + 8); a lane then holds the scores of four keys of one head, and its four
// probabilities are the B operand of O^T[dim][head] += V^T P^T (v_mfma_f32_16x16x16_bf16), whose A operand comes
// from a wave-private LDS copy of the keys' values through the transposing load. One running maximum per head and wave, moved
// only when it grows by more than 2^8. The next block's keys and values are requested before this one is computed, their
// table entries a block earlier; nothing stands between the waves until they merge, in order, at the end.
//
// What binds such a step is the chain of latencies (tile, position, table, keys) and then how long a block takes; the tile
// kernel's block was one wave's work (48 products of 32 x 32 and their LDS reads) between two barriers: four
// requests of up to 1,400 keys, 16 heads over 8 of 128 + 128 18.8 -> 11.5 us (of which about 4 are the launch), 8 heads of two
// maps over 4 of 128 + 256 31.1 -> 14.8.
//
// Places outside the visible range are read as the row's own position and their scores are masked, so no table
// entry outside it is read.
#include <math.h>

#include "common.h"
#include "mfma.h"

#define AR_WAVES 4
#define AR_KEYS 64

template <int DVB>
__global__ __launch_bounds__(AR_WAVES * 64) __attribute__((amdgpu_waves_per_eu(1, 2))) void attention_dv_rows_kernel(
    const bf16_t* __restrict__ q, int ldq, float* __restrict__ out, int ldo, const bf16_t* __restrict__ kc,
    const bf16_t* __restrict__ vc, const int* __restrict__ block_table, int max_blocks, const int* __restrict__ tiles,
    const int* __restrict__ positions, int maps, int group, int k_slots, int v_heads, int page_shift, int window, float scale,
    float softcap, float* __restrict__ partial, int per_split, int q_slots, int keep_first, const float* __restrict__ sinks,
    int chunk, const float* __restrict__ slopes) {
  constexpr int DK = 128, DV = DVB * 16, VLD = DV + 16, VP = DV / 128;  // VP: 16-byte pieces of a value row per lane
  constexpr int VS_BYTES = AR_WAVES * 16 * VLD * 2, MLD = 2 + 4 * DVB, MRG_BYTES = (AR_WAVES - 1) * 64 * MLD * 4;
  // the waves' copies of a block's values during the loop; afterwards, per lane of the waves 1..: maximum, sum, accumulators
  __shared__ __align__(16) unsigned char pool[VS_BYTES > MRG_BYTES ? VS_BYTES : MRG_BYTES];
  const int* tile = tiles + (size_t)blockIdx.y * 4;
  const int req = tile[0], row = tile[1];
  const int pos_there = positions[row], given = tile[3];
  const int pos = given >= 0 ? given : pos_there;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int sub = lane & 15, q4 = lane >> 4;
  const int ks = blockIdx.x, vh = ks / maps;  // key slot and its value head
  const int slot = (vh * group + min(sub, group - 1)) * maps + ks % maps;  // the lane's query slot
  const int first = window > 0 ? max(0, pos + 1 - window) : chunk > 0 ? pos / chunk * chunk : 0;
  const int kept = window > 0 ? min(keep_first, first) : 0;
  const int win_first = first / AR_KEYS * AR_KEYS;
  const int n_kept = min((kept + AR_KEYS - 1) / AR_KEYS, win_first / AR_KEYS);
  int it_first = 0, n_blocks = n_kept + (pos - win_first) / AR_KEYS + 1;
  auto block_keys = [&](int it) { return it < n_kept ? it * AR_KEYS : win_first + (it - n_kept) * AR_KEYS; };
  const int dv2 = DV + 2;
  float* pr = partial ? partial + (((size_t)row * q_slots + slot) * gridDim.z + blockIdx.z) * dv2 : nullptr;
  if (partial) {  // this workgroup's share of the row's blocks
    it_first = blockIdx.z * per_split;
    n_blocks = min(per_split, n_blocks - it_first);
    if (n_blocks <= 0) {  // nothing left for this split: it says so
      if (wave == 0 && q4 == 0 && sub < group) {
        pr[DV] = -INFINITY;
        pr[DV + 1] = 0.f;
      }
      return;
    }
  }
  const int* tbl = block_table + (size_t)req * max_blocks;
  const int pmask = (1 << page_shift) - 1;
  auto seen = [&](int key) { return key <= pos && (key >= first || key < kept); };
  auto there = [&](int key) { return seen(key) ? key : pos; };  // a key whose table entry may be read
  struct Pages {
    int k, v[4];
  };
  struct Turn {
    u32x4 k[4], v[4][VP];
  };
  auto ask = [&](int it, Pages& pg) {
    const int k0 = block_keys(it) + wave * 16;
    pg.k = tbl[there(k0 + sub) >> page_shift];
#pragma unroll
    for (int u = 0; u < 4; ++u) pg.v[u] = tbl[there(k0 + 4 * q4 + u) >> page_shift];
  };
  auto fetch = [&](int it, const Pages& pg, Turn& tn) {
    const int k0 = block_keys(it) + wave * 16;
    const int kk = there(k0 + sub);
    const bf16_t* kp = kc + ((((size_t)pg.k * k_slots + ks) << page_shift) + (kk & pmask)) * DK + q4 * 8;
#pragma unroll
    for (int j = 0; j < 4; ++j) tn.k[j] = *(const u32x4*)(kp + j * 32);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int kv = there(k0 + 4 * q4 + u);
      const bf16_t* vp = vc + ((((size_t)pg.v[u] * v_heads + vh) << page_shift) + (kv & pmask)) * DV + sub * 8;
#pragma unroll
      for (int c = 0; c < VP; ++c) tn.v[u][c] = *(const u32x4*)(vp + c * 128);
    }
  };
  Pages pa, pb;
  Turn ta, tb;
  ask(it_first, pa);
  u32x4 qf[4];  // B operand: head `sub`, dims 32 j + 8 q4 .. + 8
  {
    const bf16_t* qr = q + (size_t)row * ldq + (size_t)slot * DK + q4 * 8;
#pragma unroll
    for (int j = 0; j < 4; ++j) qf[j] = sub < group ? *(const u32x4*)(qr + j * 32) : u32x4{0u, 0u, 0u, 0u};
  }
  const float log2e = 1.4426950408889634f;
  const float raw_sl = softcap > 0.f ? log2e : scale * log2e;
  const float cap_in = softcap > 0.f ? 2.0f * log2e * scale / softcap : 0.f;
  const float slope2 = slopes ? slopes[slot / maps] * log2e : 0.f;
  floatx4 acc[DVB];  // O^T: dims 16 j + 4 q4 .. + 3 of head `sub`
#pragma unroll
  for (int j = 0; j < DVB; ++j) acc[j] = floatx4{0.f, 0.f, 0.f, 0.f};
  float m1 = -INFINITY, l1 = 0.f;  // of head `sub`: the wave's running maximum, and the sum over this lane's keys
  bf16_t* vw = (bf16_t*)pool + wave * 16 * VLD;
  const bf16_t* v_tr = vw + (4 * q4 + (sub >> 2)) * VLD + 4 * (sub & 3);  // what this lane names in a transposing load
  const int last = it_first + n_blocks - 1;
  fetch(it_first, pa, ta);
  ask(min(it_first + 1, last), pb);
  auto turn = [&](int it, const Turn& tn) {
    const int k0 = block_keys(it) + wave * 16;
    floatx4 sc = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < 4; ++j) sc = mfma16(tn.k[j], qf[j], sc);
    float z[4];
    float mx = -INFINITY;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int key = k0 + 4 * q4 + i;
      float x = sc[i];
      if (softcap > 0.f) x = softcap * (1.0f - 2.0f * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(x * cap_in)));
      x *= raw_sl;
      if (slopes) x += slope2 * (float)(key - pos);
      z[i] = seen(key) && sub < group ? x : -INFINITY;
      mx = fmaxf(mx, z[i]);
    }
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    if (mx > m1 + 8.0f) {  // also the first block with a visible key (m1 = -inf)
      const float alpha = exp2_diff(m1, mx);
      l1 *= alpha;
#pragma unroll
      for (int j = 0; j < DVB; ++j) acc[j] *= alpha;
      m1 = mx;
    }
    float p[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      p[i] = exp2_diff(z[i], m1);  // m1 = -inf only while no key was visible: then z is too
      l1 += p[i];
    }
    const u32x2 pk = u32x2{pack_bf16(p[0], p[1]), pack_bf16(p[2], p[3])};
    // the block's values as they lie in the cache; the wave's own LDS region, and LDS operations of one wave complete in order
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int c = 0; c < VP; ++c)  // (an infinite value times a probability of zero would be no number)
        *(u32x4*)(vw + (4 * q4 + u) * VLD + c * 128 + sub * 8) = seen(k0 + 4 * q4 + u) ? tn.v[u][c] : u32x4{0u, 0u, 0u, 0u};
#pragma unroll
    for (int j = 0; j < DVB; ++j) acc[j] = mfma16k16(lds_read_tr16(v_tr + 16 * j), pk, acc[j]);
  };
  for (int it = it_first; it <= last; it += 2) {  // two sets of registers take turns; beyond the last block: the last one again
    fetch(min(it + 1, last), pb, tb);
    ask(min(it + 2, last), pa);
    turn(it, ta);
    if (it + 1 > last) break;
    fetch(min(it + 2, last), pa, ta);
    ask(min(it + 3, last), pb);
    turn(it + 1, tb);
  }
  l1 += __shfl_xor(l1, 16, 64);
  l1 += __shfl_xor(l1, 32, 64);
  __syncthreads();  // every wave is done with its copy of the values: the memory now carries the merge
  float* mrg = (float*)pool;
  if (wave > 0) {
    float* dst = mrg + ((size_t)(wave - 1) * 64 + lane) * MLD;
    dst[0] = m1;
    dst[1] = l1;
#pragma unroll
    for (int j = 0; j < DVB; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) dst[2 + 4 * j + i] = acc[j][i];
  }
  __syncthreads();
  if (wave != 0 || sub >= group) return;
#pragma unroll
  for (int w = 0; w < AR_WAVES - 1; ++w) {
    const float* src = mrg + ((size_t)w * 64 + lane) * MLD;
    const float om = src[0], ol = src[1];
    const float mn = fmaxf(m1, om);
    const float a = exp2_diff(m1, mn), b = exp2_diff(om, mn);
    l1 = l1 * a + ol * b;
#pragma unroll
    for (int j = 0; j < DVB; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[j][i] = acc[j][i] * a + src[2 + 4 * j + i] * b;
    m1 = mn;
  }
  if (partial) {  // rows of DV + 2 floats: 8-byte aligned
#pragma unroll
    for (int j = 0; j < DVB; ++j) {
      *(float2*)(pr + 16 * j + 4 * q4) = float2{acc[j][0], acc[j][1]};
      *(float2*)(pr + 16 * j + 4 * q4 + 2) = float2{acc[j][2], acc[j][3]};
    }
    if (q4 == 0) *(float2*)(pr + DV) = float2{m1, l1};
    return;
  }
  if (sinks) l1 += __builtin_amdgcn_exp2f(sinks[slot / maps] * log2e - m1);  // one more term of the denominator
  const float inv = 1.0f / l1;
  float* o = out + (size_t)row * ldo + (size_t)slot * DV + 4 * q4;
#pragma unroll
  for (int j = 0; j < DVB; ++j) *(float4*)(o + 16 * j) = float4{acc[j][0] * inv, acc[j][1] * inv, acc[j][2] * inv, acc[j][3] * inv};
}

// The caller (attention_dv_mfma.hip) has checked the arguments; true when the sizes are taken.
bool jllm_attention_dv_rows(const void* q, int ldq, float* out, int ldo, const void* kcache, const void* vcache, const int* block_table,
                            int max_blocks, const int* tiles, int n_tiles, const int* positions, int heads, int kv_heads, int maps, int dk,
                            int dv, int page_shift, int window, float scale, float softcap, int splits, int per_split, float* partial,
                            int keep_first, const float* sinks, int chunk, const float* slopes, hipStream_t stream) {
  const int group = heads / kv_heads;
  if (dk != 128 || (dv != 128 && dv != 256) || group > 16 || ((uintptr_t)partial & 7)) return false;
  dim3 grid(kv_heads * maps, n_tiles, partial ? splits : 1);
#define AR_ARGS (const bf16_t*)q, ldq, out, ldo, (const bf16_t*)kcache, (const bf16_t*)vcache, block_table, max_blocks, tiles, positions, maps, \
                group, kv_heads * maps, kv_heads, page_shift, window, scale, softcap, partial, per_split, heads * maps, keep_first, sinks, chunk, slopes
  if (dv == 128)
    attention_dv_rows_kernel<8><<<grid, AR_WAVES * 64, 0, stream>>>(AR_ARGS);
  else
    attention_dv_rows_kernel<16><<<grid, AR_WAVES * 64, 0, stream>>>(AR_ARGS);
#undef AR_ARGS
  return true;
}
