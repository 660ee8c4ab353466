// Krylov solves of small scalar systems in one launch (rg_resident.hip).
#pragma once

#include <vector>

#include "rg_dispatch.h"
#include "rg_internal.h"

namespace rg {

// Polls of an empty slot before a workgroup of the one-launch solve gives up
// (a poll takes about a microsecond).
constexpr unsigned kResSpins = 1u << 20;

// Whether a matrix (with one method) or a batch is solved in one launch.  An
// attempt that stopped waiting (another process or stream held the GPU) costs
// up to a second: the next solve tries once more, then the launch sequence
// stays.  A refused launch is not tried again.
enum ResState { RES_UNKNOWN = 0, RES_FITS = 1, RES_OFF = 2, RES_FITS_GAVE_UP = 3 };
inline bool res_on(int state) { return state == RES_FITS || state == RES_FITS_GAVE_UP; }
enum class ResEnd { done, gave_up, refused };
inline int res_next(int state, ResEnd end)
{
    if (end == ResEnd::done) return RES_FITS;
    return end == ResEnd::gave_up && state == RES_FITS ? RES_FITS_GAVE_UP : RES_OFF;
}

// Tile sides of the one-launch solve of m with this method (Jacobi, one
// sweep); false if it does not fit in the chip's registers or the method has
// no such form.
bool resident_fits(const rg_matrix* m, int method, int (&t)[3]);
size_t resident_slot_bytes();
// Runs the Krylov loop from work->r, work->xw; work->xw is the new iterate.
// Not done (rows of xw then old or new) if the launch was refused or a
// workgroup gave up waiting for the others.
ResEnd resident_solve(rg_matrix* m, int method, const int (&t)[3], int maxit, double tol, unsigned spins,
                      KrylovState* out);

// Many independent scalar systems (full storage, one dimension, one context)
// by the textbook Jacobi-PCG in one launch.
struct ResidentBatch {
    int state = RES_UNKNOWN;
    int grid = 0;                // workgroups
    std::vector<int> tile;       // sides per system
    std::vector<int> tiles;      // tiles per system
    std::vector<int> first;      // tasks of each workgroup
    std::vector<int32_t> tasks;  // (system, rank) pairs
    void* mem = nullptr;         // device copies and slots

    ResidentBatch() = default;
    ResidentBatch(const ResidentBatch&) = delete;
    ResidentBatch& operator=(const ResidentBatch&) = delete;
    ~ResidentBatch();
    bool plan(const std::vector<rg_matrix*>& mats);
    // x from x = 0; off: the systems' offsets in dinv, b, x and the two work
    // vectors.  Not done (x then in part written) if the launch was refused or
    // a workgroup gave up.
    ResEnd solve(const std::vector<rg_matrix*>& mats, const std::vector<int64_t>& off, const double* dinv, const double* b,
               double* x, double* pub0, double* pub1, KrylovState* st, int maxit, double tol, unsigned spins,
               std::vector<KrylovState>& out);
};

}  // namespace rg
