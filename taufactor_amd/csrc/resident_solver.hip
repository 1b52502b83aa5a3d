// Resident sweep kernels of the solver kind: every compiled shape of k_resident.
#include "tauhip_resident.h"

int resident_dispatch_solver(const tf_resident& p, const ResidentArgs& a, hipStream_t st) {
    return dispatch_resident<TF_KIND_SOLVER, false>(p, a, st);
}
