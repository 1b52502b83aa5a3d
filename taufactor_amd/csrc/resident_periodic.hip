// Resident sweep kernels of the periodic kind: every compiled shape of k_resident.
#include "tauhip_resident.h"

int resident_dispatch_periodic(const tf_resident& p, const ResidentArgs& a, hipStream_t st) {
    return dispatch_resident<TF_KIND_SOLVER, true>(p, a, st);
}
