// attn_plan.hpp -- which kernel a prompt attention call of 16-bit heads takes (plain C++: host).  0: the waves of a workgroup take the 64-key blocks
// in turn, each from L2 (gqa_prefill_kernel, latent_prefill_kernel); 16 / 32: blocks of keys shared in LDS, so many rows a wave (block_attn.hpp).  A
// shared block's workgroup has four times the rows in two parts of the keys: half as many waves on a row, so a lone chain is longer, and all
// workgroups together are a quarter.
#pragma once

namespace ti {

// Grouped queries, heads of dim dims.  Waves on their own until there are two workgroups of them a CU (dims of 64: three), half as many where keys
// are few, and from 129 keys on.  us, own / 16 / 32 rows: dims of 128, 16 heads on 4, 200 rows 7.2 / 8.5, 500 11.2 / 11.5, 1000 23.4 / 18.4 / 25.6; 8
// on 2, 1000 15.8 / 17.5; 16 on 4, 20 rows behind 3000 26 / 42; 32 on 8, 256 9.3 / 8.9, 500 16.2 / 12.3 / 17.8; dims of 64, 16 on 4, 500 7.1 / 8.1,
// 2048 32 / 28 / 33; 48 on 12, 256 7.8 / 6.6.  32 rows a wave where 16 would be a second round (dims of 64, two workgroups a CU, a third: a part of a
// round of these costs less): 128, 16 on 4, 2048 rows 54 / 44; 64, 32 on 8, 1300 28.1 / 32.0, 1600 38.0 / 37.7.  Left slower than waves on their own:
// 3000 rows of 8 heads on 2 (55 / 60).
constexpr int gqa_rows_a_wave(int dim, long M, long pos0, int heads, int kv_heads) {
  const long tiles = (M + 15) / 16 * (heads / kv_heads), keys = pos0 + M;
  if (keys > 128 && tiles * kv_heads <= (keys <= 320 ? 256 : 512) + (dim == 64 ? 256 : 0)) return 0;
  return (tiles + 3) / 4 * kv_heads > (dim == 64 ? 768 : 256) ? 32 : 16;
}

// Latent heads of dim + rot dims, each with its own keys.  Waves on their own while they are at most one workgroup a CU (128 + 64: one and a half)
// from 321 keys on (128 + 64: 129), unless the heads that an XCD's run touches overflow its L2 (4 MiB; every block is then read once a wave and
// again); and where blocks of 32 rows a wave would fill a last round of workgroups, one a CU, by less than a half.  us, own / 16 / 32 rows: 128 + 64,
// 4 heads, 700 rows 14.0 / 16.8; 8, 700 15.4 / 17.1; 8, 500 behind 1000 25.4 / 30.9; 4, 1000 behind 3000 (5 MB) 100 / 71; 16, 1024 28.3 / 22.2 /
// 30.5, 2048 65 / 68 / 53; 24, 1300 48 / 51 / 57, 2048 98 / 103 / 96; 12, 3000 103 / 142 / 127; 64 + 32, 16, 300 7.6 / 7.0, 2048 42 / 33; 24, 2048 61
// / 50 / 62 (two workgroups a CU: 16 rows at any size).
constexpr int latent_rows_a_wave(int dim, int rot, long M, long pos0, int heads) {
  const bool one = dim != 64 || rot != 32;   // workgroups a CU, by their LDS
  const long keys = pos0 + M, wide = (M + 127) / 128 * heads, rounds = (wide + 255) / 256;
  const int touched = heads == 1 ? 1 : heads / 8 + (heads % 8 ? 2 : 0);   // heads in an eighth of the (head, rows) list
  const bool l2 = touched * keys * (2 * dim + rot) * 2 <= 4l << 20;
  const bool large = dim == 128 && rot == 64;
  if (keys > (large ? 128 : 320) &&
      (((M + 15) / 16 * heads <= (large && keys > 320 ? 384 : 256) && l2) || (one && wide > 256 && 3 * 256 * rounds >= 4 * wide))) return 0;
  return one && (M + 63) / 64 * heads > 256 ? 32 : 16;
}

}  // namespace ti
