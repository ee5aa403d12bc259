// coarse.hpp -- the bottom of the V-cycle as one launch (coarse.hip).
#pragma once
#include "solver.hpp"

namespace hpcgx
{

// Sections of a row's entries: left of the diagonal, right of it, of these the
// ones outside and inside the last colour, and the row as a whole.
enum CoarseSection : int
{
    SEC_LOWER = 0,
    SEC_UPPER = 1,
    SEC_MID = 2,
    SEC_TAIL = 3,
    SEC_ROW = 4,
    SEC_COUNT = 5
};

// One step of a symmetric Gauss-Seidel sweep over a level: some rows of one
// colour, and the slot groups (of four) its one or two sums take.
struct CoarseStep
{
    int kind;       // CoarseKind
    int off, n;     // rows [off, off + n), at most a team's threads
    int va, ia, na; // first sum: its first group among the values and among the
                    // columns (section * groups + group), and how many
    int vb, ib, nb; // second sum
};

// What one workgroup needs of a level, in device memory (coarse_build).
struct CoarseLevel
{
    const void* val;           // values, and diagonal
    const void* dg;
    const int32_t* diag_idx;   // slot of the diagonal
    const uint2* at;           // LDS byte offsets of the columns' x, 16 bits each: [section][group][row]
    const int32_t* f2c_fine;   // to the next level
    const int32_t* f2c_coarse;
    const CoarseStep* steps;   // pre-smoothing steps, then post-smoothing ones
    void* r;                   // the level's vectors (level 0: given with the launch)
    void* x;
    int m, mc, npre, npost;
    int whole_rows;            // the post-smoother has steps of kind CK_FWD_T
    int lds_x, lds_t;          // where the level's x and t lie in LDS (bytes)
};

// One V-cycle from lv[0] down over nl levels: x = M^-1 r.
struct CoarseRun
{
    const CoarseLevel* lv;
    int nl;
    int r_f64;                 // r is f64 whatever the vector type
    const void* r;
    void* x;
    const int* gate;
};

// Where the parts of a plan's allocation lie, in bytes: the columns, from 0, then
// the steps, then the descriptions, which hold pointers and start where those may
// (the bottom of an eight-colour hierarchy has 15 steps of 36 bytes).
struct CoarseLayout
{
    size_t steps, levels, bytes;
};

inline CoarseLayout coarse_layout(size_t ncolumns, size_t nsteps, size_t nlevels)
{
    auto up = [](size_t at, size_t a) { return (at + a - 1) / a * a; };
    CoarseLayout o;
    o.steps = up(sizeof(uint16_t) * ncolumns, alignof(CoarseStep));
    o.levels = up(o.steps + sizeof(CoarseStep) * nsteps, alignof(CoarseLevel));
    o.bytes = o.levels + sizeof(CoarseLevel) * nlevels;
    return o;
}

// build the plans of a problem whose levels and vectors exist; they are complete,
// and CoarsePlan::upload done with, when P.s has been waited for
int coarse_build(Problem& P);
void coarse_free(Problem& P);
// the first level that runs in one workgroup, with everything below it
// (nlevels: none)
int coarse_first(const Problem& P, Prec prec);
CoarseRun coarse_run(const Problem& P, int l, Prec prec, const void* r, bool r_f64, void* x, const int* gate);
int launch_coarse(const CoarseRun& run, Prec prec, size_t lds, hipStream_t s);
// the same for `n` problems, one workgroup each (runs in device memory)
int launch_coarse_batch(const CoarseRun* runs, int n, Prec prec, size_t lds, hipStream_t s);

}  // namespace hpcgx
