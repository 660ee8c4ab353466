// Krylov solves of small scalar systems in one launch (rg_resident.hip).
#pragma once

#include "rg_dispatch.h"
#include "rg_internal.h"

namespace rg {

// Polls of an empty slot before a workgroup of the one-launch solve gives up
// (a poll takes about a microsecond).
constexpr unsigned kResSpins = 1u << 20;

// Tile sides of the one-launch solve of m with this method (Jacobi, one
// sweep); false if it does not fit in the chip's registers or the method has
// no such form.
bool resident_fits(const rg_matrix* m, int method, int (&t)[3]);
// As resident_fits, for any grid: at most `rows` nodes and `cells` padded
// cells per tile, at most `tiles` tiles.
bool resident_tiles(int dim, const int64_t* nn, int rows, int cells, int tiles, int (&t)[3]);
size_t resident_slot_bytes();
// Runs the Krylov loop from work->r, work->xw; work->xw is the new iterate.
// False (xw then any iterate) if the launch was refused or a workgroup gave
// up waiting for the others.
bool resident_solve(rg_matrix* m, int method, const int (&t)[3], int maxit, double tol, unsigned spins,
                    KrylovState* out);

}  // namespace rg
