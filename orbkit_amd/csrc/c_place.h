// Which MO coefficients the lanes of the FP64 fused kernel (fused_f64.h) read
// for each accumulator and K step.  Plain integer arithmetic: the same functions
// run on the host, where a test walks every place against the bounds of C.
#pragma once

namespace okmi_fused {

// Groups of 4 MOs of the instance that a pass runs, from the groups asked for:
// every count for rho and rho with first derivatives of standard bases (l <= 3,
// real spherical or Cartesian rows), and up to 10 for the pass of seven AO sets;
// multiples of 4 for the others; MO values: every second count.
// C may be read where the caller has it, with no padding after it: an instance
// of NT tiles of 16 MOs and NR groups of 4 must hold an MO in the last of them,
// so that only that one is partly empty (last_tile_mo, last_group_mo).
__host__ __device__ inline int f64_units(int u, int pass, bool standard, bool mo)
{
    if (!standard || pass == 2 || pass == 3) return pass == 4 && u > 8 ? u : (u + 3) & ~3;
    return mo && u > 2 ? (u + 1) & ~1 : u;
}

// MO within the last of NT tiles of 16 that lane n16 = 0 .. 15 reads, and within
// the last of NR groups of 4 (after the tiles) that lane n4 = 0 .. 3 reads; `last`:
// the last MO in memory, which the places past it repeat
__host__ __device__ inline int last_tile_mo(int n16, int last, int NT)
{
    const int most = last - 16 * (NT - 1);
    return n16 < most ? n16 : most > 0 ? most : 0;
}
__host__ __device__ inline int last_group_mo(int n4, int last, int NT, int NR)
{
    const int most = last - 16 * NT - 4 * (NR - 1);
    return n4 < most ? n4 : most > 0 ? most : 0;
}

// Row of a shell of N rows that place w = 0 .. W - 1 gives to the K step of rows
// R .. R + W - 1 (the W lane groups of split_rows); places past the last row
// repeat it
template <int W> __host__ __device__ constexpr int split_row(int R, int w, int N)
{
    return R + W <= N ? R + w : R + w < N ? R + w : N - 1;
}

}  // namespace okmi_fused
