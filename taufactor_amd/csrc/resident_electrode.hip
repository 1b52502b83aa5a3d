// Resident sweep kernels of the electrode kind (closed and periodic y/z): every compiled shape of k_resident.
#include "tauhip_resident.h"

int resident_dispatch_electrode(const tf_resident& p, const ResidentArgs& a, int periodic, hipStream_t st) {
    return periodic ? dispatch_resident<TF_KIND_ELECTRODE, true>(p, a, st)
                    : dispatch_resident<TF_KIND_ELECTRODE, false>(p, a, st);
}
