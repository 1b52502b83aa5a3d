// Sweep kernels of the uneven batch for 4 to 6 half-sweeps (sweep_batch.hip).
#include "tauhip_sweep.h"

int sweep_dispatch_batch_deep(int H, BatchArgs& a, int nw, int rpw, hipStream_t st) {
    switch (H) {
        case 4: return dispatch_batch_shape<4>(a, nw, rpw, st);
        case 5: return dispatch_batch_shape<5>(a, nw, rpw, st);
        case 6: return dispatch_batch_shape<6>(a, nw, rpw, st);
        default: return fail(-1, "n_half=%d out of range 1..%d", H, TF_MAX_FUSED_HALF_SWEEPS);
    }
}
