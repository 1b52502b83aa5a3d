// Resident sweep kernels of the per-voxel diffusivity kind: every compiled shape of k_resident.
#include "tauhip_resident.h"

int resident_dispatch_field(const tf_resident& p, const ResidentArgs& a, hipStream_t st) {
    return dispatch_resident<TF_KIND_FIELD, false>(p, a, st);
}
