// Sweep kernels of the Solver kind (register-blocked): every compiled shape of
// k_sweep for 1 to 3 half-sweeps; the deeper ones, as long to compile, are in
// sweep_solver_deep.hip.
#include "tauhip_sweep.h"

int sweep_dispatch_solver_deep(int H, SweepArgs& a, int B, int nw, int rpw, hipStream_t st);

int sweep_dispatch_solver(int H, SweepArgs& a, int B, int nw, int rpw, hipStream_t st) {
    switch (H) {
        case 1: return dispatch_shape<1, TF_KIND_SOLVER>(a, B, nw, rpw, st);
        case 2: return dispatch_shape<2, TF_KIND_SOLVER>(a, B, nw, rpw, st);
        case 3: return dispatch_shape<3, TF_KIND_SOLVER>(a, B, nw, rpw, st);
        default: return sweep_dispatch_solver_deep(H, a, B, nw, rpw, st);
    }
}
