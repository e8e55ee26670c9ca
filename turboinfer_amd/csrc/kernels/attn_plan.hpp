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

}  // namespace ti
