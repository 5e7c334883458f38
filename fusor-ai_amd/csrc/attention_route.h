// Which of the int8 attention's two paths a call takes, from its sizes alone (plain C++).
#pragma once

#include <algorithm>
#include <cmath>
#include <cstddef>

namespace fg {

// Whether a call is the faster in the one launch of attention_fused.hip (head_dim at most 128)
// than a unit ((image, head)) at a time. The one launch walks a row's blocks of 32 keys in order,
// so few rows over many keys leave the chip idle behind that chain; a unit at a time pays two
// launches per unit but spreads its keys.
//
// Both sides in microseconds, fitted to 6500 calls drawn over 1 to 64 units, 1 to 4096 queries, 16 to
// 16384 keys, both exponentials and 28 head sizes. A block's cost is that of the kernel's records
// (blocks of 32 channels, eights of channels in the last): four blocks of channels, and three with
// a tail of 24, run one block of keys at a time, the others two. Of the 6500 calls 14 take more than
// 5 % longer on the side chosen here than unit by unit (most of them calls of 50 to 60 us; the
// longest chains of one query up to 1.29 times), and 69 more than 5 % longer than on the faster
// side. One launch against unit by unit, measured: heads of 64, 6 units x 1024 queries x 1024 keys
// 76 and 109, 1 unit of the same 75 and 56, 12 units x 1024 x 4096 256 and 371, 12 units x 1 x 4096
// 249 and 210; heads of 128, 3 units x 1024 x 512 86 and 72, 6 x 1024 x 1024 145 and 123; heads of
// 116, 3 x 426 x 533 98 and 65; heads of 88, 3 x 483 x 483 85 and 68.
inline bool attend_in_one_launch(size_t images, size_t heads, size_t head_dim, size_t queries, size_t keys, bool fast)
{
    static const double kBlock[4][4] = {
        {1.08, 1.14, 1.17, 1.19}, {1.60, 1.65, 1.89, 1.70}, {2.02, 2.09, 3.30, 2.11}, {3.18, 3.40, 4.21, 3.73}};
    const size_t pb = (head_dim + 31) / 32, tail = (head_dim - 32 * (pb - 1) + 7) / 8;
    const double u = double(images * heads), k = double(keys), q = double(queries), hd = double(head_dim);
    const double waves = u * std::ceil(q / 32);  // 1024 SIMDs
    const double block = (kBlock[pb - 1][tail - 1] + (fast ? 0.0 : 0.47)) * std::max(1.0, 0.7 * waves / 1024);
    const double fused = 27 + std::ceil(k / 32) * block;
    const double steps = 46 + 4.7 * u + 1.65e-4 * k * hd + u * k * (0.002 + 2.75e-6 * q);
    return fused <= steps;
}

}  // namespace fg
