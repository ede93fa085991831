// Estimated times of the products of more than 64 rows (kernels/ops.py: `_tile_us` and `_wide_us`, whose constants come with every
// call) and the walks over their choices: some eighty per product and tile count, which a prompt of a length that was not seen before
// waits for: us for the four products of the 0.6B shape at 487, 833 and 1,500 rows, walked in Python 420, 422 and 260, here 110, 118 and
// 65; at a length with the tiles of one that was seen 45, 51 and 40 / 12, 12 and 7.
#include <algorithm>
#include <cmath>
#include <limits>

#include "host_core.h"

namespace {

int64_t up(int64_t a, int64_t b) { return (a + b - 1) / b; }

int64_t across(const JllmTileKind& k, int64_t N, bool gated) { return up(N, gated ? k.columns / 2 : k.columns); }

// workgroups with K whole
int64_t groups(const JllmTileKind& k, int64_t M, int64_t N, bool gated) {
  const int64_t a = across(k, N, gated);
  return k.wide_last ? M / k.rows * a + up(a, 2) : a * up(M, k.rows);
}

double norm_us(const JllmTileRules& r, int64_t M, int64_t N) { return r.norm_us + r.norm_element_us * (double)M * (double)N; }

double tile_us(const JllmTileRules& r, const JllmTileKind& k, int64_t M, int64_t N, int64_t K, bool gated, int64_t cut) {
  const double cus = r.cus;
  const int64_t steps = up(K, 64 * cut), most = k.two ? 2 * r.cus : r.cus, all = groups(k, M, N, gated) * cut;
  const int64_t rounds = all / most, last = all % most;
  double t = (double)rounds * ((double)steps * (k.two ? k.all : k.full) + k.round_us);
  const double step = last > r.cus ? k.few + (k.all - k.few) * (double)(last - r.cus) / cus : k.lone + (k.full - k.lone) * (double)last / cus;
  if (last) t += (double)steps * step + k.round_us;
  if (k.wide_last) t += r.wide_extra[M % k.rows > 64] * (double)steps * (rounds ? k.full : step);
  t = k.fixed + std::hypot(t, (double)N * (double)K * (gated ? 4.0 : 2.0) / r.bytes_per_us);
  return cut > 1 ? t + (r.cut_us + r.cut_element_us * (double)M * (double)N * (double)cut) : t;
}

void weigh(JllmTileChoice& best, double us, const JllmTileKind& k, int64_t cut) {
  if (us < best.us) best = JllmTileChoice{us, k.code, (int32_t)cut};
}

double stream_us(const JllmStreamRules& r, int64_t M, int64_t N, int64_t K, bool gated, int rows, int tile, int parts) {
  const int64_t groups = up(N, gated ? rows / 2 : rows) * up(M, tile) * parts;
  const double step = (double)(up(K / 128, parts) * 2) * (r.block_us + r.block_row_us * ((rows + tile) / 8.0 - 12.0));
  double t;
  if (tile == 64) {  // two on a compute unit
    const int64_t full = groups / (2 * (int64_t)r.cus), last = groups % (2 * (int64_t)r.cus);
    t = (double)full * step * r.pair_all;
    if (last) t += last <= r.cus ? step : step * (r.pair_few + (r.pair_all - r.pair_few) * (double)(last - r.cus) / r.cus);
  } else {
    t = (double)up(groups, r.cus) * step;
  }
  t = std::max(t, (double)N * (double)K * (gated ? 4.0 : 2.0) / r.bytes_per_us) + (tile == 64 ? r.fixed_64 : r.fixed_128);
  if (parts > 1) t += r.merge_us + r.merge_kb_us * parts * rows * (double)std::min<int64_t>(tile, M) * 4 / 1024;
  return t;
}

}  // namespace

extern "C" {

double jllm_stream_us(const JllmStreamRules* rules, int M, int N, int K, int gated, int rows, int tile, int parts) {
  return stream_us(*rules, M, N, K, gated != 0, rows, tile, parts);
}

void jllm_stream_tiles(const JllmStreamRules* rules, int M, int N, int K, int gated, int32_t* plan) {
  const JllmStreamRules& r = *rules;
  double best = std::numeric_limits<double>::infinity();
  plan[0] = plan[1] = 64, plan[2] = 1;
  const int64_t blocks = K / 128;
  for (int rows = 32; rows <= 128; rows += 32)
    for (int tile = 64; tile <= 128; tile += 64) {
      const int64_t tiles = up(N, gated ? rows / 2 : rows) * up(M, tile);
      for (int parts = 1; parts <= 4; ++parts) {
        const int64_t per = up(blocks, parts);
        if (parts > 1 && (tiles * parts > 2 * (int64_t)r.cus || per < r.least_blocks || up(blocks, per) != parts)) continue;
        const double t = stream_us(r, M, N, K, gated != 0, rows, tile, parts);
        if (t < best) best = t, plan[0] = rows, plan[1] = tile, plan[2] = parts;
      }
    }
}

double jllm_tile_us(const JllmTileRules* rules, int kind, int M, int N, int K, int gated, int cut) {
  if (kind < 0 || kind >= rules->n_small + rules->n_large || cut < 1) return -1.0;
  return tile_us(*rules, rules->kinds[kind], M, N, K, gated != 0, cut);
}

void jllm_small_tiles(const JllmTileRules* rules, int M, int N, int K, int gated, JllmTileChoice* out) {
  const JllmTileRules& r = *rules;
  const double norm = norm_us(r, M, N);
  const int64_t stages = K / 64;
  out[0] = out[1] = JllmTileChoice{std::numeric_limits<double>::infinity(), r.fallback, 1};
  for (int i = 0; i < r.n_small; ++i) {
    const JllmTileKind& k = r.kinds[i];
    if (gated && k.plain_only) continue;
    const int64_t whole = groups(k, M, N, gated != 0);
    for (int c = 0; c < r.n_small_cuts; ++c) {
      const int64_t cut = r.small_cuts[c];
      if (cut > 1 && (gated || K / cut < r.small_part || whole * cut > 3 * (int64_t)r.cus || stages <= up(stages, cut) * (cut - 1))) continue;
      const double t = tile_us(r, k, M, N, K, gated != 0, cut);
      weigh(out[0], t, k, cut);
      weigh(out[1], cut == 1 ? t + norm : t, k, cut);
    }
  }
}

void jllm_large_tiles(const JllmTileRules* rules, int M, int N, int K, int gated, int normed, JllmTileChoice* best) {
  const JllmTileRules& r = *rules;
  const double norm = normed ? norm_us(r, M, N) : 0.0;
  for (int i = r.n_small; i < r.n_small + r.n_large; ++i) {
    const JllmTileKind& k = r.kinds[i];
    if (k.wide_last && (M % k.rows == 0 || M % k.rows > 128)) continue;
    for (int64_t cut = 1; cut <= (gated ? 1 : r.large_cuts); ++cut) {
      if (cut > 1 && K / cut < r.large_part) break;
      if (k.odd_cuts && (cut == 1 || cut == 2 || cut == 4)) continue;
      const double t = tile_us(r, k, M, N, K, gated != 0, cut);
      weigh(*best, cut == 1 ? t + norm : t, k, cut);
    }
  }
}
}
