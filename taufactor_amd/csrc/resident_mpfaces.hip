// Resident sweep kernels of the MultiPhase kind read through face codes: every compiled shape of k_resident.
#include "tauhip_resident.h"

int resident_dispatch_mpfaces(const tf_resident& p, const ResidentArgs& a, hipStream_t st) {
    return dispatch_resident<TF_KIND_MULTIPHASE_FACES, false>(p, a, st);
}
