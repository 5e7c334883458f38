// Which kernel a T2b128 product of more than 16 rows takes, from its sizes alone (plain C++).
#pragma once

namespace fg {

constexpr int kT2Rows = 64, kT2Cols = 128;  // a staged workgroup's tile

// Workgroups of t2_lds_kernel for `rows` rows and `outputs` columns.
inline long t2_staged_groups(long rows, long outputs)
{
    return (outputs + kT2Cols - 1) / kT2Cols * ((rows + kT2Rows - 1) / kT2Rows);
}

// Whether a product of `groups` groups of 128 inputs is the faster on the staged tiles (t2_lds_kernel)
// than on a wave per tile of 32 rows (t2_gemm_kernel).
//   About a workgroup per CU, from where the staged tiles' traffic and not one workgroup's chain of
//   stages (1 us a group) is what counts: 4096 x 14336 at 96 rows (224 workgroups) 36 us against 40,
//   1024 x 4096 at 512 rows (256) 13.1 against 18.8, at 256 rows (128) 12.5 against 10.8, 896 x 4864 at
//   256 rows (152) 11.4 against 11.7, 4864 x 896 at 1024 rows (112) 48 against 29.
//   32 rows would leave half of each tile empty. So do 65 to 96 rows of the second tiles, and up to
//   about a workgroup per CU the chain is as long for them: there the fewer the rows past 64 and the deeper the
//   product, the later the staged tiles are the faster (past 96 groups the other kernel's waves of more
//   columns fall behind by themselves). 8192 x 12800 at 65, 80 and 96 rows (200 workgroups) 78, 77 and 77
//   against 60, 62 and 66; 8192 x 14336 (224) 79, 77 and 77 against 66, 68 and 74; 4096 x 12800 37, 35 and
//   35 against 33, 35 and 35; 2048 x 14336 21, 21 and 20 against 20, 22 and 23; 14336 x 16384 at 65 rows
//   136 against 151; 8192 x 22016 at 65 rows (344) 84 against 93. Over 828 products measured with both,
//   of 33 to 2048 rows, 1 to 112 groups and 200 workgroups or more, the side taken is at most 4 % the slower.
inline bool t2_takes_staged(long rows, long outputs, long groups)
{
    const long staged = t2_staged_groups(rows, outputs);
    if (rows <= 32 || staged < 200) return false;
    if (rows <= 64 || rows > 96 || staged >= 300 || groups <= 8) return true;
    if (staged < 220) return groups < 40 && rows >= 88;
    return groups > 96 || rows >= (groups < 40 ? 72 : 92);
}

}  // namespace fg
