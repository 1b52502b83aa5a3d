// Sweep kernels of the Solver kind for 4 to 6 half-sweeps (sweep_solver.hip).
#include "tauhip_sweep.h"

int sweep_dispatch_solver_deep(int H, SweepArgs& a, int B, int nw, int rpw, hipStream_t st) {
    switch (H) {
        case 4: return dispatch_shape<4, TF_KIND_SOLVER>(a, B, nw, rpw, st);
        case 5: return dispatch_shape<5, TF_KIND_SOLVER>(a, B, nw, rpw, st);
        case 6: return dispatch_shape<6, TF_KIND_SOLVER>(a, B, nw, rpw, st);
        default: return fail(-1, "n_half=%d out of range 1..%d", H, TF_MAX_FUSED_HALF_SWEEPS);
    }
}
