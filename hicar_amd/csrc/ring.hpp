// Ring conditions (icar_adv_apply_bc) of one species: bc_x 1 copies column
// nx-2 into the last column, 2 wraps both columns; bc_y 2 wraps both rows.
// The rule is x sides first, then y sides, whose corners copy what the x sides
// wrote.  Both are one pass here: the x sides skip the rows the y sides write,
// and the y sides read a corner's value where the x sides would have copied it
// from, so no cell is read that another thread writes.
#pragma once
#include "common.hpp"

namespace icaradv {

// threads of the x and the y sides, each a multiple of 256
__host__ __device__ inline unsigned ring_x_threads(const Dims &d, int bc_x)
{
    return bc_x ? ((unsigned)d.ny * (unsigned)d.nz + 255u) / 256u * 256u : 0u;
}
__host__ __device__ inline unsigned ring_y_threads(const Dims &d, int bc_y)
{
    return bc_y == 2 ? ((unsigned)d.nx * (unsigned)d.nz + 255u) / 256u * 256u : 0u;
}

// thread t of the ring_x_threads + ring_y_threads of the species q (E: a
// 4- or 2-byte word; the stored bits are copied)
template <typename E>
__device__ __forceinline__ void ring_cells(E *__restrict__ q, const Dims &d, unsigned t, int bc_x,
                                           int bc_y)
{
    const unsigned nxt = ring_x_threads(d, bc_x);
    if (t < nxt) {
        const int k = (int)(t % (unsigned)d.nz), j = (int)(t / (unsigned)d.nz);
        if (j >= d.ny || (bc_y == 2 && (j == 0 || j == d.ny - 1))) return;
        q[ix(d, d.nx - 1, k, j)] = q[ix(d, bc_x == 1 ? d.nx - 2 : 1, k, j)];
        if (bc_x == 2) q[ix(d, 0, k, j)] = q[ix(d, d.nx - 2, k, j)];
    } else {
        t -= nxt;
        const int i = (int)(t % (unsigned)d.nx), k = (int)(t / (unsigned)d.nx);
        if (bc_y != 2 || k >= d.nz) return;
        int s = i;  // the column the x sides copy i from
        if (bc_x && i == d.nx - 1) s = bc_x == 1 ? d.nx - 2 : 1;
        if (bc_x == 2 && i == 0) s = d.nx - 2;
        q[ix(d, i, k, 0)] = q[ix(d, s, k, d.ny - 2)];
        q[ix(d, i, k, d.ny - 1)] = q[ix(d, s, k, 1)];
    }
}

}  // namespace icaradv
