// attn_plan.hpp -- which kernel a prompt attention call of 16-bit heads takes (plain C++: host).
#pragma once

namespace ti {

// 0: the waves of a workgroup take the 64-key blocks in turn, each from L2 (gqa_prefill_kernel, latent_prefill_kernel); 16 / 32: blocks of keys
// shared in LDS, so many rows a wave (block_attn.hpp). A shared block's workgroup has four times the rows in two parts of the keys: half as many
// waves on a row, so a lone chain is longer, and all workgroups together are a quarter. Times are of calls as a prompt's layers make them: keys and
// values just written by another kernel, the caches full of other data (with keys in the L2s waves on their own are up to 40 % faster, shared blocks
// 5 %).

// Grouped queries, heads of dim dims. us, own / 16 / 32 rows: dims of 128, 16 heads on 4, 40 rows 8.8 / 7.5, 500 13.5 / 13.2, 1000 27.1 / 21.2 /
// 28.6, 1300 37.3 / 40.7 / 35.2, 2048 59.0 / 59.3 / 46.9; 8 on 2, 300 12.4 / 11.2, 1000 20.2 / 20.1, 200 behind 2000 34.6 / 38.5 (whole prompts of 6
// layers, own -> 16 rows: 4 on 1, 600 354 -> 341, 20 on 5, 64 behind 1000 634 -> 605, 30 behind 1800 604 -> 572: their keys come from farther still);
// dims of 64, 16 on 4, 300 8.1 / 7.7, 500 8.7 / 9.3, 1000 14.1 / 14.4, 2048 36.1 / 29.2 / 35.6; 4 on 1, 2048 19.8 / 23.2; 48 on 12, 256 8.5 / 7.0,
// 800 32.9 / 23.1 / 27.0; 32 on 8, 1300 38.8 / 30.6 / 33.5, 1600 50.6 / 40.7 / 39.8 (prompts, own -> 16: 12 on 3, 30 behind 1800 288 -> 306). So:
// heads of 64 dims' waves on their own where keys are many and they are at most three workgroups a CU; 32 rows a wave where 16 would be a second
// round (64: two workgroups a CU, a third round). Left slower than waves on their own: 3000 rows of 16 heads on 4 of 128 (108 / 119, a second round
// that is half full).
constexpr int gqa_rows_a_wave(int dim, long M, long pos0, int heads, int kv_heads) {
  const long tiles = (M + 15) / 16 * (heads / kv_heads);
  if (dim == 64 && pos0 + M > 320 && tiles * kv_heads <= 768) return 0;
  return (tiles + 3) / 4 * kv_heads > (dim == 64 ? 768 : 256) ? 32 : 16;
}

// Latent heads of dim + rot dims, each with its own keys: all of them new to the caches. us, own / 16 / 32 rows: 128 + 64, 4 heads, 40 rows 11.0 /
// 6.5, 640 22.5 / 16.2; 8, 16 behind 1000 29.8 / 20.1, 500 behind 1000 45 / 31; 16, 1000 34 / 23 / 31, 1300 46 / 46 / 39, 2048 68 / 70 / 55; 24, 1300
// 55 / 57 / 63, 2048 100 / 106 / 97; 12, 3000 105 / 150 / 134; 40, 1300 79 / 91 / 71; 64 + 64, 16, 1000 24.5 / 16.4 / 21.4, 2048 49 / 49 / 38; 64 +
// 32, 16, 2048 47 / 32 / 36, 40 107 / 80 / 97. So: shared blocks, 16 rows a wave while they are one round of a workgroup a CU, else 32 (64 + 32: LDS
// for two a CU, 16 at any size); waves on their own where 32 rows fill the last round by less than a half of it.
constexpr int latent_rows_a_wave(int dim, int rot, long M, int heads) {
  if ((M + 63) / 64 * heads <= 256 || (dim == 64 && rot == 32)) return 16;
  const long wide = (M + 127) / 128 * heads, rounds = (wide + 255) / 256;
  return rounds > 1 && 3 * 256 * rounds >= 4 * wide ? 0 : 32;
}

}  // namespace ti
