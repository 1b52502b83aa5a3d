// Sweep kernels of the uneven batch (k_sweep_batch, k_sweep_batch_queue) for
// 1 to 3 half-sweeps; the deeper ones, as long to compile, are in
// sweep_batch_deep.hip.
#include "tauhip_sweep.h"

int sweep_dispatch_batch_deep(int H, BatchArgs& a, int nw, int rpw, hipStream_t st);

int sweep_dispatch_batch(int H, BatchArgs& a, int nw, int rpw, hipStream_t st) {
    switch (H) {
        case 1: return dispatch_batch_shape<1>(a, nw, rpw, st);
        case 2: return dispatch_batch_shape<2>(a, nw, rpw, st);
        case 3: return dispatch_batch_shape<3>(a, nw, rpw, st);
        default: return sweep_dispatch_batch_deep(H, a, nw, rpw, st);
    }
}
