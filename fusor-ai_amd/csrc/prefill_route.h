// Which kernels a prefill chunk's attention takes in parallel order, from its sizes alone (plain C++).
#pragma once

namespace fg {

// Whether attn_flash_kernel takes a chunk of n rows whose last sees kmax keys (heads of 32, 64 or 128);
// rows_fit: attn_rows_kernel's LDS holds the scores of its blocks of rows. Four layers' reads in
// microseconds, attn_flash_kernel against the others:
//   few keys: one launch instead of two (the chunk's rows kept, then the attention). 14 heads of 64, from
//   position 64: 1, 2, 4 and 8 rows 190, 204, 213 and 229 against 181, 190, 201 and 224, break even near
//   145 keys under 8 rows and 110 from there; 64 rows from position 0 234 against 226, from 30 235 against
//   237; heads of 128, 8 rows from 128 270 against 259, break even near 160, 96 rows from position 0 277
//   against 269, 128 rows 292 against 296;
//   more keys than attn_rows_kernel holds: its two substitutes spread a row's keys over workgroups
//   where the flash kernel's eight waves walk them, so their time grows with the rows times the
//   heads and its own does not until the chip is full. On 461 such chunks of 32 to 512 rows, 2 to
//   32 heads over 1 to 16, the line below is at most 8 % off the faster side: 32 rows from 6500, 7 heads of
//   128 over 1, 1447 against 846; 64 rows from 5000, 4 heads of 64 over 4, 684 against 620, 96 rows 689
//   against 922; 4 heads of 32 over 1, 32 rows from 7000 587 against 495. Under
//   32 rows the substitutes are kept: 16 rows from 3500, heads of 64, 386 against 535.
// Otherwise the flash kernel: 4 rows from 2000, heads of 64, 362 against 708. (5 to 16 rows of a model of 128
// hidden values are bound by the host's launches, not by these kernels: up to about 450 keys the second launch is
// their 7 %, 257 against 241. From 512 hidden values on the kernels are what counts: 8 rows over 160 keys, heads of 32,
// 158 against 176, of 64 207 against 221, of 128 310 against 310.)
inline bool prefill_takes_flash(int D, int heads, int kv_heads, int n, int kmax, bool rows_fit)
{
    if (!rows_fit) return n >= 32 && (long long)n * (heads * D + 64 * kv_heads) >= 540ll * D;
    const int few = D == 128 ? (n < 32 ? 160 : 112) : n < 8 ? 144 : n < 32 ? 112 : 64;
    return kmax > few;
}

}  // namespace fg
