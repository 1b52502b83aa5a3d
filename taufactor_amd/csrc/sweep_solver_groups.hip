// Sweep kernels of the Solver kind with its codes in groups of four rows.
#include "tauhip_sweep.h"

int sweep_dispatch_solver_groups(int H, SweepArgs& a, int B, int nw, int rpw, hipStream_t st) {
    return dispatch_groups<TF_KIND_SOLVER_GROUPS>(H, a, B, nw, rpw, st);
}
