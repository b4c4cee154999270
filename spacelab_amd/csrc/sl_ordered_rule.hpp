// Which launch shape of the ordered pair pass a size takes when none is chosen (host code).
#pragma once

namespace sl {

// An index into SL_ORD_SHAPES (sl_kernels_ordered.hip).  Timed at 27 sizes from 2 to 40,000
// balls of aggregates on MI355X (us per step, the shape taken first):
//   <= 256     8 wavefronts with batches of 32 partners: a batch for each up to 256 partners
//              (129 balls 8.2; with batches of 64 8.6)
//   <= 512     2 balls a workgroup, 8 wavefronts, a CU for each of up to 256 workgroups (512 balls
//              12.3; 4 balls 12.6)
//   <= 1,024   4 balls, likewise (1,000 balls 18.3; 2 balls in 4 wavefronts 21.5)
//   <= 1,536   2 balls in 4 wavefronts, three workgroups a CU hold them all at once (1,500 balls
//              30.4; 4 balls 35.1)
//   <= 20,000  4 balls, 4 wavefronts, no scan for contacts first (2,200 balls 54.9, with the scan
//              58.9; 1,800 42.6 and 42.9; 5,000 161 and 181)
//   above      8 balls: fewer adds per pair (20,000 balls 1,977 and, 4 balls, 2,024; 40,000 7,585
//              and 7,857; 12,000 to 25,000 differ by less than 3%, either way)
inline int ordered_default_shape(int n)
{
    return n <= 256 ? 7 : n <= 512 ? 0 : n <= 1024 ? 1 : n <= 1536 ? 5 : n <= 20000 ? 3 : 4;
}

}  // namespace sl
