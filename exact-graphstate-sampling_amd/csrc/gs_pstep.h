// Descriptor of a pair of steps as the in-place engine's chain sweep uses it (gs_pair.hip).
#pragma once
#include "gs_pair.h"

namespace gs {

// Coordinates: with 8-byte entries 0 is the unit bit 0 (one aligned run of 2 per thread); then 8 of the threads, the
// blocks', the tiles'.  None of the run's and the threads' changes step k+1's slot index.
struct PStep {
    PairDesc d;
    uint64_t off[4], g1;       // step k's offsets; step k+1's g
    uint32_t t0m, t1m, parm;   // step k's routing, a bit per offset
    uint32_t u0m, u1m, uparm;  // step k+1's
    int m1, ntq;
    int lg_grid, lg_iter, xcd;
};

}  // namespace gs
